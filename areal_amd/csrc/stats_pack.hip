// Data movement and logging reductions either side of the loss: packing padded [B, S] batches
// into the packed layout by cu_seqlens and back, re-aligning a packed batch, and the masked
// sum / count / min / max of many per-token statistics in one launch.
//
// Follows areal/utils/data.py: pack_tensor_dict (:496-545), pad_packed_tensor_dict (:822-982),
// unpack_sequence + pad_and_stack_tensors_along_first_dim as used by reorder_and_pad_outputs
// (areal/engine/core/train_engine.py:110-144); and areal/utils/stats_tracker.py: _avg_of,
// _min_of, _max_of (:455-560), which reduce every logged tensor under its denominator mask.
#include "common.hpp"

#include <algorithm>

namespace {

constexpr int PK_THREADS = 256;
// Blocks of a launch: HIP runs one of 2^32 threads or more without its last blocks, and without an error.
constexpr int64_t PK_MAX_BLOCKS = ((int64_t)1 << 32) / PK_THREADS - 1;

// 16 bytes at any address. The compiler picks the access the target allows for the alignment
// (gfx950 runs with unaligned access enabled, where this is still one 16-byte instruction).
// (A vector, not a struct: predicated copies of a struct went through LDS.)
typedef uint32_t Bytes16 __attribute__((ext_vector_type(4), aligned(1)));

// number of nonzero bytes among the four of x
DEVI int nonzero_bytes(uint32_t x) {
  x = (x | (x >> 4)) & 0x0f0f0f0fu;
  x = (x | (x >> 2)) & 0x03030303u;
  x = (x | (x >> 1)) & 0x01010101u;
  return __popc(x);
}

// lens[b] = number of nonzero entries of mask row b (one block per row), 16 mask bytes per load. host (nullable, host
// memory): the same numbers.
__global__ __launch_bounds__(PK_THREADS) void rowlens_kernel(const uint8_t* mask, int64_t S,
                                                             int32_t* lens, double* host) {
  __shared__ int sm[4];
  const uint8_t* row = mask + (int64_t)blockIdx.x * S;
  int len = 0;
  const int64_t n16 = S >> 4;
  for (int64_t i = threadIdx.x; i < n16; i += blockDim.x) {
    const Bytes16 v = *(const Bytes16*)(row + 16 * i);
#pragma unroll
    for (int k = 0; k < 4; ++k) len += nonzero_bytes(v[k]);
  }
  for (int64_t s = 16 * n16 + threadIdx.x; s < S; s += blockDim.x) len += row[s] != 0;
  len = wave_sum(len);
  if ((threadIdx.x & 63) == 0) sm[threadIdx.x >> 6] = len;
  __syncthreads();
  if (threadIdx.x == 0) {
    len = sm[0] + sm[1] + sm[2] + sm[3];
    lens[blockIdx.x] = len;
    if (host != nullptr) host[blockIdx.x] = (double)len;
  }
}

// Inclusive prefix sum over the wave's 64 lanes: inside each row of 16 through DPP, then the
// totals of the rows to the left (lanes 15, 31, 47) are added.
DEVI int wave_inclusive_sum(int v) {
  v += dpp_move<DPP_ROW_SHR + 1>(0, v);
  v += dpp_move<DPP_ROW_SHR + 2>(0, v);
  v += dpp_move<DPP_ROW_SHR + 4>(0, v);
  v += dpp_move<DPP_ROW_SHR + 8>(0, v);
  const int t0 = lane_value(v, 15), t1 = lane_value(v, 31), t2 = lane_value(v, 47);
  const int row = (threadIdx.x & 63) >> 4;
  return v + (row == 0 ? 0 : row == 1 ? t0 : row == 2 ? t0 + t1 : t0 + t1 + t2);
}

// cu = exclusive prefix sums of lens, *max_len = max(lens) (one block; 4 entries per thread and
// round, two barriers per round). host (nullable, host memory): the total and the longest.
constexpr int SCAN_ITEMS = 4;
__global__ __launch_bounds__(PK_THREADS) void cu_scan_kernel(const int32_t* lens, int64_t B,
                                                             int32_t* cu, int32_t* max_len, double* host) {
  __shared__ int sm_sum[PK_THREADS / 64], sm_max[PK_THREADS / 64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  int carry = 0, mx = 0;
  if (threadIdx.x == 0) cu[0] = 0;
  for (int64_t b0 = 0; b0 < B; b0 += PK_THREADS * SCAN_ITEMS) {
    const int64_t b = b0 + (int64_t)threadIdx.x * SCAN_ITEMS;
    int len[SCAN_ITEMS];
#pragma unroll
    for (int i = 0; i < SCAN_ITEMS; ++i) len[i] = b + i < B ? lens[b + i] : 0;
    int tot = 0;
#pragma unroll
    for (int i = 0; i < SCAN_ITEMS; ++i) { tot += len[i]; mx = len[i] > mx ? len[i] : mx; }
    const int incl = wave_inclusive_sum(tot);
    __syncthreads();  // the previous round's readers are done
    if (lane == 63) sm_sum[w] = incl;
    __syncthreads();
    int base = carry + incl - tot;
    for (int i = 0; i < w; ++i) base += sm_sum[i];
#pragma unroll
    for (int i = 0; i < SCAN_ITEMS; ++i) {
      base += len[i];
      if (b + i < B) cu[b + i + 1] = base;
    }
    for (int i = 0; i < PK_THREADS / 64; ++i) carry += sm_sum[i];
  }
  mx = wave_reduce(mx, [](int a, int b) { return a > b ? a : b; });
  __syncthreads();
  if (lane == 0) sm_max[w] = mx;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int i = 1; i < PK_THREADS / 64; ++i) mx = sm_max[i] > mx ? sm_max[i] : mx;
    *max_len = mx;
    if (host != nullptr) {
      host[0] = (double)carry;
      host[1] = (double)mx;
    }
  }
}

// One integer of a queued call's results to host memory, for a caller that looks there until it has arrived.
__global__ void int_to_host_kernel(const int32_t* x, double* host) { host[0] = (double)*x; }

// Copy of n contiguous bytes by the whole block: 16 bytes per thread and access, whatever the
// two addresses' alignment, four loads in flight per thread before the first store. A run whose
// length is not a multiple of 16 ends with a piece that overlaps its predecessor (the same bytes twice).
// Bound by the latency of its loads (a block moves 16 KiB at most): they are issued without a predicate,
// at clamped indices. With a predicate each, every load was waited for before the next was issued:
// unpacking 557 Ki tokens of 4 bytes into 256 rows took 18.0 us and takes 4.4, packing six tensors of them
// 21.9 and 9.4.
template <int THREADS>
DEVI void copy_bytes(char* dst, const char* src, int64_t n, int thread) {
  if (n < 16) {
    if ((int64_t)thread < n) dst[thread] = src[thread];
    return;
  }
  const int64_t pieces = (n + 15) >> 4;
  for (int64_t i0 = thread; i0 < pieces; i0 += 4 * THREADS) {
    Bytes16 v[4];
    int64_t at[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int64_t o = 16 * (i0 + u * THREADS);
      at[u] = o < n - 16 ? o : n - 16;
      v[u] = *(const Bytes16*)(src + at[u]);
    }
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (i0 + u * THREADS < pieces) *(Bytes16*)(dst + at[u]) = v[u];
  }
}
DEVI void block_copy_bytes(char* dst, const char* src, int64_t n) { copy_bytes<PK_THREADS>(dst, src, n, threadIdx.x); }

// Several tensors packed in one launch. Block (c, k) writes packed tokens [c * chunk, (c + 1) *
// chunk) of tensor k: it finds the sequence of its first token (every wave searches cu_seqlens
// with 64 probes per round) and then walks the sequences its chunk touches, each one contiguous
// run of a padded row to one contiguous run of the packed array. No block is empty. The chunk is at
// most 16 KiB of the widest tensor and 2048 tokens, a thread has four loads of 16 bytes in flight at once.
constexpr int PK_MAX_TENSORS = 8;
constexpr int PK_CHUNK_BYTES = 16384, PK_CHUNK_MAX = 2048;
struct PackArgs {
  const char* src[PK_MAX_TENSORS];
  char* dst[PK_MAX_TENSORS];
  int64_t eb[PK_MAX_TENSORS];  // bytes of one token's trailing dimensions
  const int32_t* cu;
  int n_seqs;
  int64_t S, total;
  int chunk;  // tokens per block
};
// BY_WAVE: a chunk's sequences go to the block's four waves in turn, 63 of them known from one load of cu_seqlens (see
// pack_plan). Bound by the latency of cu_seqlens and the copies for short rows, by HBM from 2 Mi tokens on.
template <bool BY_WAVE>
__global__ __launch_bounds__(PK_THREADS) void pack_rows_kernel(PackArgs a) {
  const int k = blockIdx.y;
  int64_t t = (int64_t)blockIdx.x * a.chunk;
  const int64_t t1 = t + a.chunk < a.total ? t + a.chunk : a.total;
  // (selects, not an index into the argument arrays: those would be copied to scratch memory)
  const char* src = a.src[0]; char* dst = a.dst[0]; int64_t eb = a.eb[0];
#pragma unroll
  for (int i = 1; i < PK_MAX_TENSORS; ++i)
    if (k == i) { src = a.src[i]; dst = a.dst[i]; eb = a.eb[i]; }
  // sequence of token t: the number of sequence ends at or before it (same value in every wave)
  int b = wave_count_le(a.cu + 1, a.n_seqs, t, threadIdx.x & 63);
  if constexpr (BY_WAVE) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    for (; b < a.n_seqs; b += 63) {
      const int entry = a.cu[b + lane < a.n_seqs ? b + lane : a.n_seqs];
      const int n = a.n_seqs - b < 63 ? a.n_seqs - b : 63;
      for (int i = wave; i < n; i += PK_THREADS / 64) {
        const int64_t start = lane_value(entry, i), end = lane_value(entry, i + 1);
        if (start >= t1) return;
        const int64_t from = start > t ? start : t, stop = end < t1 ? end : t1;
        if (stop > from)
          copy_bytes<64>(dst + from * eb, src + ((int64_t)(b + i) * a.S + (from - start)) * eb, (stop - from) * eb, lane);
      }
      if (lane_value(entry, n) >= t1) return;
    }
    return;
  }
  while (t < t1 && b < a.n_seqs) {
    const int64_t start = a.cu[b], end = a.cu[b + 1];
    const int64_t stop = end < t1 ? end : t1;
    if (stop > t) block_copy_bytes(dst + t * eb, src + ((int64_t)b * a.S + (t - start)) * eb, (stop - t) * eb);
    t = stop > t ? stop : t;
    ++b;
  }
}

// Fill pattern of n <= 16 bytes. When n divides 16 the words hold it repeated (16-byte stores).
// (Words selected, not bytes indexed: an indexed argument would be copied to scratch memory.)
struct Fill { uint32_t w[4]; int n; };
DEVI char fill_byte(const Fill& f, int i) {
  const uint32_t x = i < 8 ? (i < 4 ? f.w[0] : f.w[1]) : (i < 12 ? f.w[2] : f.w[3]);
  return (char)(x >> (8 * (i & 3)));
}

// n bytes at dst (the start of an element) filled with the pattern by the whole block: 16-byte
// stores of the repeated pattern when its length divides 16, byte by byte otherwise and at the end.
DEVI void block_fill_bytes(char* dst, int64_t n, const Fill& f) {
  int64_t done = 0;
  if ((16 % f.n) == 0) {
    Bytes16 pat;
#pragma unroll
    for (int w = 0; w < 4; ++w) pat[w] = f.w[w];
    const int64_t n16 = n >> 4;
    for (int64_t i = threadIdx.x; i < n16; i += blockDim.x) *(Bytes16*)(dst + 16 * i) = pat;
    done = 16 * n16;
  }
  for (int64_t i = done + threadIdx.x; i < n; i += blockDim.x) dst[i] = fill_byte(f, (int)(i % f.n));
}

// Tokens per block of the row-wise kernels below: 16 KiB of an element, at most 2048 tokens.
static int64_t pk_chunk_tokens(int64_t eb) {
  const int64_t c = PK_CHUNK_BYTES / eb;
  return c < 1 ? 1 : (c > PK_CHUNK_MAX ? PK_CHUNK_MAX : c);
}

// How pack_rows_kernel cuts `total` tokens of `rows` rows. By waves unless a token is wider than 512 bytes: the whole block
// copies one run after the other, each with its latency, and has most threads idle on runs of under 4 KiB. Six tensors
// (25 B a token), whole block / waves, us: 1024 rows of mean 105 17.1 / 5.6, 64 of 105 13.7 / 3.7, 1024 of 271 12.5 / 7.5,
// 512 of 1062 10.5 / 7.9, 256 of 2175 9.8 / 7.8, 512 of 4351 21.1 / 19.2 (5.8 TB/s); wide tokens: 64 rows of 530 x 512 B
// 8.5 / 8.6, of 530 x 4 KiB 42.8 / 44.3, 8 of 158 x 4 KiB 3.9 / 4.4.
// Chunks of four runs (two, four, eight, sixteen: 64 rows of mean 66 3.0, 3.6, 4.0, 5.0; 1024 of 271 9.1, 7.9, 7.4, 7.4; 512 of
// 756 7.9, 6.4, 7.7, 7.7; only 1024 of 74 prefers eight, 5.4 for 7.8), and few rather than full ones while
// there are less than 128 (8 rows of 4351: 3.3 for 4.1); smaller ones otherwise cost their start (512 of 4351 in 512s 34.2).
struct PackPlan { bool by_wave; int64_t chunk; };
static PackPlan pack_plan(int64_t rows, int64_t total, int64_t max_eb) {
  const int64_t whole = pk_chunk_tokens(max_eb);
  if (max_eb > 512) return {false, whole};
  const int64_t runs = round_up_i64(4 * (total / rows + 1), 64), spread = round_up_i64(total / 128 + 1, 256);
  // (a launch takes less than 2^24 blocks of 256 threads: more than 67 million rows of a few tokens each)
  return {true, std::max(std::min(whole, std::min(runs, spread)), total / (1 << 23) + 1)};
}

// padded[row][j] = j < len_b ? packed[cu[b] + j] : fill, b = row_seq[row] (or row). Block
// (row, c) writes tokens [c * chunk, (c + 1) * chunk) of its row: one contiguous copy, one fill.
__global__ __launch_bounds__(PK_THREADS) void unpack_kernel(const char* packed, char* padded,
                                                            const int32_t* cu, const int32_t* row_seq,
                                                            int64_t S, int64_t eb, Fill fill, int chunks,
                                                            int chunk) {
  const int64_t row = blockIdx.x / chunks;
  const int64_t j0 = (int64_t)(blockIdx.x % chunks) * chunk;
  const int64_t nj = S - j0 < chunk ? S - j0 : chunk;
  const int64_t b = row_seq ? row_seq[row] : row;  // packed sequence shown in this row
  const int64_t start = cu[b], len = (int64_t)cu[b + 1] - start;
  int64_t ncopy = len - j0;
  ncopy = ncopy < 0 ? 0 : (ncopy > nj ? nj : ncopy);
  char* d = padded + (row * S + j0) * eb;
  if (ncopy > 0) block_copy_bytes(d, packed + (start + j0) * eb, ncopy * eb);
  if (ncopy < nj) block_fill_bytes(d + ncopy * eb, (nj - ncopy) * eb, fill);
}

// unpack_kernel where a row's sequence is given as rows[row] = {first packed token, length}: one read, which may go to
// host memory. (The pattern is an argument: of a constant the compiler makes a byte loop, 15 us in place of 4.)
__global__ __launch_bounds__(PK_THREADS) void unpack_rows_kernel(const char* packed, char* padded, const u32x2* rows,
                                                                 int64_t S, int64_t eb, Fill fill, int chunks, int chunk) {
  const int64_t row = blockIdx.x / chunks;
  const int64_t j0 = (int64_t)(blockIdx.x % chunks) * chunk;
  const int64_t nj = S - j0 < chunk ? S - j0 : chunk;
  const u32x2 seq = rows[row];
  int64_t ncopy = (int64_t)seq[1] - j0;
  ncopy = ncopy < 0 ? 0 : (ncopy > nj ? nj : ncopy);
  char* d = padded + (row * S + j0) * eb;
  if (ncopy > 0) block_copy_bytes(d, packed + ((int64_t)seq[0] + j0) * eb, ncopy * eb);
  if (ncopy < nj) block_fill_bytes(d + ncopy * eb, (nj - ncopy) * eb, fill);
}

// dst[cu_new[s] + j] = j < old length of s ? src[cu_old[s] + j] : fill; sequences of cu_new
// beyond n_old (a trailing pad segment) are all fill. arange != 0: dst is int64 position ids,
// and the fill is j (position inside the new sequence, src == NULL) or j - old length instead.
// Block c writes tokens [c * chunk, (c + 1) * chunk) of dst, sequence by sequence as pack_rows_kernel.
__global__ __launch_bounds__(PK_THREADS) void realign_kernel(const char* src, char* dst,
                                                             const int32_t* cu_old, int n_old,
                                                             const int32_t* cu_new, int n_new,
                                                             int64_t eb, Fill fill, int arange,
                                                             int64_t total_new, int chunk) {
  int64_t t = (int64_t)blockIdx.x * chunk;
  const int64_t t1 = t + chunk < total_new ? t + chunk : total_new;
  int s = wave_count_le(cu_new + 1, n_new, t, threadIdx.x & 63);
  while (t < t1 && s < n_new) {
    const int64_t start = cu_new[s], end = cu_new[s + 1];
    const int64_t stop = end < t1 ? end : t1;
    if (stop > t) {
      const int64_t j0 = t - start, j1 = stop - start;  // positions inside the new sequence
      const int64_t len = (s < n_old && src != nullptr) ? (int64_t)cu_old[s + 1] - cu_old[s] : 0;
      const int64_t jc = j1 < len ? j1 : len;            // copied positions are [j0, jc)
      if (jc > j0) block_copy_bytes(dst + t * eb, src + ((int64_t)cu_old[s] + j0) * eb, (jc - j0) * eb);
      const int64_t jf = j0 > len ? j0 : len;            // filled positions are [jf, j1)
      if (jf < j1) {
        char* d = dst + (start + jf) * eb;
        if (arange) {
          const int64_t shift = src == nullptr ? 0 : (s < n_old ? (int64_t)cu_old[s + 1] - cu_old[s] : 0);
          const int64_t per = eb >> 3;  // int64 channels per token
          for (int64_t i = threadIdx.x; i < (j1 - jf) * per; i += blockDim.x)
            ((int64_t*)d)[i] = jf + i / per - shift;
        } else {
          block_fill_bytes(d, (j1 - jf) * eb, fill);
        }
      }
      t = stop;
    }
    ++s;
  }
}

// A packed batch with one more sequence behind it: block (c, k) writes tokens [c * chunk, (c + 1) * chunk)
// of tensor k, those below `total` copied, the rest filled (arange: 0, 1, 2, ... in the int64 channels
// of a token). No sequence moves, so nothing is searched; the first block also writes the two
// cu_seqlens arrays. One launch: six tensors of 557 Ki tokens took six launches of 20 us, this 6.7 us.
struct PadArgs {
  const char* src[PK_MAX_TENSORS];
  char* dst[PK_MAX_TENSORS];
  int64_t eb[PK_MAX_TENSORS];
  Fill fill[PK_MAX_TENSORS];
  int arange;  // bit k: tensor k
  const int32_t* cu;
  int32_t* cu_copy;
  int32_t* cu_new;
  int n_seqs, n_tensors;
  int64_t total, total_new;
  int chunk;
  double* host_total;  // nullable, pinned host memory: receives cu[n_seqs]
};
__global__ __launch_bounds__(PK_THREADS) void pad_packed_kernel(PadArgs a) {
  const int k = blockIdx.y;
  if (k == 0 && blockIdx.x == 0) {
    if (threadIdx.x == 0 && a.host_total != nullptr) *a.host_total = (double)a.cu[a.n_seqs];
    for (int i = threadIdx.x; i <= a.n_seqs; i += PK_THREADS) {
      const int32_t c = a.cu[i];
      a.cu_copy[i] = c;
      a.cu_new[i] = c;
    }
    if (threadIdx.x == 0) a.cu_new[a.n_seqs + 1] = (int32_t)a.total_new;
  }
  if (k >= a.n_tensors) return;
  const char* src = a.src[0]; char* dst = a.dst[0]; int64_t eb = a.eb[0];
  uint32_t f0 = a.fill[0].w[0], f1 = a.fill[0].w[1], f2 = a.fill[0].w[2], f3 = a.fill[0].w[3];
  int fn = a.fill[0].n;
#pragma unroll
  for (int i = 1; i < PK_MAX_TENSORS; ++i)
    if (k == i) {
      src = a.src[i]; dst = a.dst[i]; eb = a.eb[i];
      f0 = a.fill[i].w[0]; f1 = a.fill[i].w[1]; f2 = a.fill[i].w[2]; f3 = a.fill[i].w[3];
      fn = a.fill[i].n;
    }
  const int64_t t0 = (int64_t)blockIdx.x * a.chunk;
  const int64_t t1 = t0 + a.chunk < a.total_new ? t0 + a.chunk : a.total_new;
  const int64_t tc = t1 < a.total ? t1 : a.total, tf = t0 > a.total ? t0 : a.total;
  if (t0 < tc) block_copy_bytes(dst + t0 * eb, src + t0 * eb, (tc - t0) * eb);
  if (tf < t1) {
    if ((a.arange >> k) & 1) {
      const int64_t per = eb >> 3;  // int64 channels per token
      for (int64_t i = threadIdx.x; i < (t1 - tf) * per; i += PK_THREADS)
        ((int64_t*)(dst + tf * eb))[i] = tf - a.total + i / per;
    } else {
      block_fill_bytes(dst + tf * eb, (t1 - tf) * eb, Fill{{f0, f1, f2, f3}, fn});
    }
  }
}

// ---------------------------------------------------------------------------------------
// Masked statistics of K tensors in one launch.
// ---------------------------------------------------------------------------------------
constexpr int STATS_MAX_K = 32;
constexpr int STATS_BLOCKS = 256;
struct StatsArgs {
  const float* v[STATS_MAX_K];
  const uint8_t* m[STATS_MAX_K];  // denominator mask of tensor k (null: all ones)
  int K;
  int64_t n;
};
struct StatPart { double sum, cnt; float mn, mx; };

DEVI double block_sum_d(double v, double* smem) {
  v = wave_sum(v);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  __syncthreads();
  if (lane == 0) smem[w] = v;
  __syncthreads();
  double r = 0.0;
  for (int i = 0; i < (int)(blockDim.x >> 6); ++i) r += smem[i];
  return r;
}
DEVI float block_minmax(float v, float* smem, bool is_min) {
  v = is_min ? wave_min(v) : wave_max(v);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  __syncthreads();
  if (lane == 0) smem[w] = v;
  __syncthreads();
  float r = smem[0];
  for (int i = 1; i < (int)(blockDim.x >> 6); ++i) r = is_min ? fminf(r, smem[i]) : fmaxf(r, smem[i]);
  return r;
}

// grid (STATS_BLOCKS, K): partial over a slice of tensor blockIdx.y
__global__ __launch_bounds__(PK_THREADS) void stats_partial_kernel(StatsArgs a, StatPart* parts) {
  __shared__ double sm_d[4];
  __shared__ float sm_f[4];
  const int k = blockIdx.y;
  const float* v = a.v[k];
  const uint8_t* m = a.m[k];
  double sum = 0.0, cnt = 0.0;
  float mn = pos_inf(), mx = neg_inf();
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < a.n;
       i += (int64_t)gridDim.x * blockDim.x) {
    if (m != nullptr && m[i] == 0) continue;
    const float x = v[i];
    sum += (double)x; cnt += 1.0;
    mn = fminf(mn, x); mx = fmaxf(mx, x);
  }
  sum = block_sum_d(sum, sm_d);
  cnt = block_sum_d(cnt, sm_d);
  mn = block_minmax(mn, sm_f, true);
  mx = block_minmax(mx, sm_f, false);
  if (threadIdx.x == 0) parts[(int64_t)k * gridDim.x + blockIdx.x] = StatPart{sum, cnt, mn, mx};
}
// out[k] = {sum, count, min, max} (min = +inf, max = -inf when the mask is empty)
__global__ __launch_bounds__(PK_THREADS) void stats_final_kernel(const StatPart* parts, int nparts,
                                                                 double* out) {
  __shared__ double sm_d[4];
  __shared__ float sm_f[4];
  const int k = blockIdx.x;
  double sum = 0.0, cnt = 0.0;
  float mn = pos_inf(), mx = neg_inf();
  for (int i = threadIdx.x; i < nparts; i += blockDim.x) {
    const StatPart p = parts[(int64_t)k * nparts + i];
    sum += p.sum; cnt += p.cnt; mn = fminf(mn, p.mn); mx = fmaxf(mx, p.mx);
  }
  sum = block_sum_d(sum, sm_d);
  cnt = block_sum_d(cnt, sm_d);
  mn = block_minmax(mn, sm_f, true);
  mx = block_minmax(mx, sm_f, false);
  if (threadIdx.x == 0) {
    out[4 * k] = sum; out[4 * k + 1] = cnt; out[4 * k + 2] = (double)mn; out[4 * k + 3] = (double)mx;
  }
}

bool make_fill(const void* fill, int fill_bytes, Fill& f) {
  if (fill_bytes < 0 || fill_bytes > 16) return false;
  f.n = fill_bytes > 0 ? fill_bytes : 1;
  for (int i = 0; i < 4; ++i) f.w[i] = 0;
  if (fill_bytes > 0 && fill != nullptr)
    for (int i = 0; i < 16; ++i)  // (a length that does not divide 16: the words past it are not read)
      f.w[i >> 2] |= (uint32_t)((const uint8_t*)fill)[i % fill_bytes] << (8 * (i & 3));
  return true;
}

}  // namespace

extern "C" {

// attention_mask [B, S] bytes (nonzero = token) -> lens [B], cu_seqlens [B+1], *max_len, all
// int32 on the device (data.py:513-517).
static int seqlens_from_mask(const uint8_t* attention_mask, int64_t B, int64_t S, int32_t* lens, int32_t* cu_seqlens,
                             int32_t* max_len, double* host, double* host_lens, hipStream_t stream) {
  if (B < 0 || S < 0) return AREAL_ERR_BAD_ARG;
  if (!cu_seqlens || !max_len || (B > 0 && (!attention_mask || !lens))) return AREAL_ERR_BAD_ARG;
  if (B > PK_MAX_BLOCKS || B * S >= ((int64_t)1 << 31)) return AREAL_ERR_UNSUPPORTED;
  if (B > 0) {
    hipLaunchKernelGGL(rowlens_kernel, dim3((unsigned)B), dim3(PK_THREADS), 0, stream,
                       attention_mask, S, lens, host_lens);
    AREAL_CHECK_LAUNCH();
  }
  hipLaunchKernelGGL(cu_scan_kernel, dim3(1), dim3(PK_THREADS), 0, stream, lens, B, cu_seqlens,
                     max_len, host);
  AREAL_CHECK_LAUNCH();
  return AREAL_OK;
}

int areal_seqlens_from_mask_ex(const uint8_t* attention_mask, int64_t B, int64_t S, int32_t* lens,
                               int32_t* cu_seqlens, int32_t* max_len, double* host, hipStream_t stream) {
  return seqlens_from_mask(attention_mask, B, S, lens, cu_seqlens, max_len, host, nullptr, stream);
}

int areal_seqlens_from_mask_rows(const uint8_t* attention_mask, int64_t B, int64_t S, int32_t* lens,
                                 int32_t* cu_seqlens, int32_t* max_len, double* host_lens, hipStream_t stream) {
  return seqlens_from_mask(attention_mask, B, S, lens, cu_seqlens, max_len, nullptr, host_lens, stream);
}

int areal_seqlens_from_mask(const uint8_t* attention_mask, int64_t B, int64_t S, int32_t* lens,
                            int32_t* cu_seqlens, int32_t* max_len, hipStream_t stream) {
  return areal_seqlens_from_mask_ex(attention_mask, B, S, lens, cu_seqlens, max_len, nullptr, stream);
}

int areal_int_to_host(const int32_t* value, double* host, hipStream_t stream) {
  if (!value || !host) return AREAL_ERR_BAD_ARG;
  hipLaunchKernelGGL(int_to_host_kernel, dim3(1), dim3(1), 0, stream, value, host);
  AREAL_CHECK_LAUNCH();
  return AREAL_OK;
}

// packed [total, E] <- the first len_b tokens of every row of padded [B, S, E]; elem_bytes = bytes
// of one token's trailing dimensions (data.py:535-541). Up to 8 tensors of one batch (host
// arrays of device pointers and of element sizes) in one launch.
int areal_pack_padded_multi(const void* const* padded, void* const* packed, const int64_t* elem_bytes,
                            int n_tensors, const int32_t* cu_seqlens, int64_t B, int64_t S,
                            int64_t total, hipStream_t stream) {
  if (B < 0 || S < 0 || total < 0 || n_tensors < 0 || n_tensors > PK_MAX_TENSORS) return AREAL_ERR_BAD_ARG;
  if (total == 0 || n_tensors == 0) return AREAL_OK;
  if (!padded || !packed || !elem_bytes || !cu_seqlens || B == 0) return AREAL_ERR_BAD_ARG;
  PackArgs a;
  for (int k = 0; k < PK_MAX_TENSORS; ++k) { a.src[k] = nullptr; a.dst[k] = nullptr; a.eb[k] = 0; }
  for (int k = 0; k < n_tensors; ++k) {
    if (!padded[k] || !packed[k] || elem_bytes[k] <= 0) return AREAL_ERR_BAD_ARG;
    a.src[k] = (const char*)padded[k]; a.dst[k] = (char*)packed[k]; a.eb[k] = elem_bytes[k];
  }
  int64_t max_eb = 1;
  for (int k = 0; k < n_tensors; ++k) max_eb = elem_bytes[k] > max_eb ? elem_bytes[k] : max_eb;
  const auto [by_wave, chunk] = pack_plan(B, total, max_eb);
  const int64_t chunks = ceil_div_i64(total, chunk);
  if (chunks > PK_MAX_BLOCKS || B > (1 << 30)) return AREAL_ERR_UNSUPPORTED;
  a.cu = cu_seqlens; a.n_seqs = (int)B; a.S = S; a.total = total; a.chunk = (int)chunk;
  const dim3 grid((unsigned)chunks, (unsigned)n_tensors);
  hipLaunchKernelGGL((by_wave ? pack_rows_kernel<true> : pack_rows_kernel<false>), grid, dim3(PK_THREADS), 0, stream, a);
  AREAL_CHECK_LAUNCH();
  return AREAL_OK;
}

int areal_pack_padded(const void* padded, void* packed, const int32_t* cu_seqlens, int64_t B,
                      int64_t S, int64_t elem_bytes, int64_t total, hipStream_t stream) {
  if (elem_bytes <= 0) return AREAL_ERR_BAD_ARG;
  if (total > 0 && (!padded || !packed)) return AREAL_ERR_BAD_ARG;
  return areal_pack_padded_multi(&padded, &packed, &elem_bytes, 1, cu_seqlens, B, S, total, stream);
}

// padded [B, S, E] <- packed sequences, the rest filled with the fill pattern (fill_bytes <= 16
// bytes repeated over the element; NULL = zero bytes): unpack_sequence + reorder_list +
// pad_and_stack. row_seq [B] (nullable): row r shows packed sequence row_seq[r].
int areal_unpack_to_padded(const void* packed, void* padded, const int32_t* cu_seqlens,
                           const int32_t* row_seq, int64_t B, int64_t S, int64_t elem_bytes,
                           const void* fill, int fill_bytes, hipStream_t stream) {
  if (B < 0 || S < 0 || elem_bytes <= 0) return AREAL_ERR_BAD_ARG;
  if (B == 0 || S == 0) return AREAL_OK;
  if (!padded || !cu_seqlens) return AREAL_ERR_BAD_ARG;
  Fill f;
  if (!make_fill(fill, fill_bytes, f)) return AREAL_ERR_BAD_ARG;
  const int64_t chunk = pk_chunk_tokens(elem_bytes), chunks = ceil_div_i64(S, chunk);
  if (chunks * B > PK_MAX_BLOCKS) return AREAL_ERR_UNSUPPORTED;
  hipLaunchKernelGGL(unpack_kernel, dim3((unsigned)(chunks * B)), dim3(PK_THREADS), 0, stream,
                     (const char*)packed, (char*)padded, cu_seqlens, row_seq, S, elem_bytes, f, (int)chunks,
                     (int)chunk);
  AREAL_CHECK_LAUNCH();
  return AREAL_OK;
}

// areal_unpack_to_padded whose rows are given as {first packed token, length} pairs and end in zeros. The pairs may lie in
// pinned host memory (which has to stay until the launch has finished); a block reads one of them.
int areal_unpack_rows(const void* packed, void* padded, const uint32_t* rows, int64_t B, int64_t S, int64_t elem_bytes,
                      hipStream_t stream) {
  if (B < 0 || S < 0 || elem_bytes <= 0) return AREAL_ERR_BAD_ARG;
  if (B == 0 || S == 0) return AREAL_OK;
  if (!padded || !rows) return AREAL_ERR_BAD_ARG;
  const int64_t chunk = pk_chunk_tokens(elem_bytes), chunks = ceil_div_i64(S, chunk);
  if (chunks * B > PK_MAX_BLOCKS) return AREAL_ERR_UNSUPPORTED;
  hipLaunchKernelGGL(unpack_rows_kernel, dim3((unsigned)(chunks * B)), dim3(PK_THREADS), 0, stream, (const char*)packed,
                     (char*)padded, (const u32x2*)rows, S, elem_bytes, Fill{{0u, 0u, 0u, 0u}, 16}, (int)chunks, (int)chunk);
  AREAL_CHECK_LAUNCH();
  return AREAL_OK;
}

// Re-layout of a packed batch (data.py:848-911, :927-969): sequence s moves from cu_old to
// cu_new (new length >= old length, the tail filled); cu_new may hold extra trailing
// sequences (the batch pad), filled entirely. position_ids != 0: elem_bytes is a multiple of 8
// (int64 channels); src == NULL writes 0..len-1 per new sequence, otherwise the pads continue
// with 0, 1, 2, ... after the copied part.
int areal_realign_packed(const void* src, void* dst, const int32_t* cu_old, int64_t n_old,
                         const int32_t* cu_new, int64_t n_new, int64_t elem_bytes,
                         const void* fill, int fill_bytes, int position_ids, int64_t total_new,
                         hipStream_t stream) {
  if (n_old < 0 || n_new < 0 || elem_bytes <= 0 || total_new < 0) return AREAL_ERR_BAD_ARG;
  if (total_new == 0) return AREAL_OK;
  if (!dst || !cu_new || n_new == 0 || (n_old > 0 && !cu_old)) return AREAL_ERR_BAD_ARG;
  if (position_ids && (elem_bytes % 8 != 0 || ((uintptr_t)dst & 7))) return AREAL_ERR_ALIGNMENT;
  if (!position_ids && src == nullptr && n_old > 0) return AREAL_ERR_BAD_ARG;
  Fill f;
  if (!make_fill(fill, fill_bytes, f)) return AREAL_ERR_BAD_ARG;
  const int64_t chunk = pk_chunk_tokens(elem_bytes), chunks = ceil_div_i64(total_new, chunk);
  if (chunks > PK_MAX_BLOCKS || n_new > (1 << 30)) return AREAL_ERR_UNSUPPORTED;
  hipLaunchKernelGGL(realign_kernel, dim3((unsigned)chunks), dim3(PK_THREADS), 0, stream,
                     (const char*)src, (char*)dst, cu_old, (int)n_old, cu_new, (int)n_new,
                     elem_bytes, f, position_ids, total_new, (int)chunk);
  AREAL_CHECK_LAUNCH();
  return AREAL_OK;
}

// A packed batch padded to total_new > total tokens by one more sequence (data.py:927-969), up to 8
// tensors (host arrays) in one launch: dst[k] [total_new] <- src[k] [total], the rest filled with
// fills[16 k .. 16 k + fill_bytes[k]) repeated, or, where position_ids[k] != 0 (elem_bytes a multiple of
// 8), with 0, 1, 2, ... cu_copy [n_seqs + 1] <- cu_seqlens, cu_new [n_seqs + 2] <- cu_seqlens, total_new.
int areal_pad_packed_multi(const void* const* src, void* const* dst, const int64_t* elem_bytes, const void* fills,
                           const int* fill_bytes, const int* position_ids, int n_tensors,
                           const int32_t* cu_seqlens, int64_t n_seqs, int32_t* cu_copy, int32_t* cu_new,
                           int64_t total, int64_t total_new, hipStream_t stream) {
  return areal_pad_packed_multi_ex(src, dst, elem_bytes, fills, fill_bytes, position_ids, n_tensors, cu_seqlens, n_seqs,
                                   cu_copy, cu_new, total, total_new, nullptr, stream);
}
// ... and cu_seqlens[n_seqs] to pinned host memory (nullable), for a caller that took `total` from the tensors' shapes.
int areal_pad_packed_multi_ex(const void* const* src, void* const* dst, const int64_t* elem_bytes, const void* fills,
                              const int* fill_bytes, const int* position_ids, int n_tensors,
                              const int32_t* cu_seqlens, int64_t n_seqs, int32_t* cu_copy, int32_t* cu_new,
                              int64_t total, int64_t total_new, double* host_total, hipStream_t stream) {
  if (n_tensors < 0 || n_tensors > PK_MAX_TENSORS || n_seqs < 0 || total < 0 || total_new <= total)
    return AREAL_ERR_BAD_ARG;
  if (!cu_seqlens || !cu_copy || !cu_new) return AREAL_ERR_BAD_ARG;
  if (n_tensors > 0 && (!src || !dst || !elem_bytes || !fills || !fill_bytes || !position_ids)) return AREAL_ERR_BAD_ARG;
  if (n_seqs > (1 << 30) || total_new >= ((int64_t)1 << 31)) return AREAL_ERR_UNSUPPORTED;
  PadArgs a{};
  int64_t max_eb = 1;
  for (int k = 0; k < n_tensors; ++k) {
    if (!dst[k] || elem_bytes[k] <= 0 || (total > 0 && !src[k])) return AREAL_ERR_BAD_ARG;
    if (position_ids[k]) {
      if (elem_bytes[k] % 8 != 0 || ((uintptr_t)dst[k] & 7)) return AREAL_ERR_ALIGNMENT;
      a.arange |= 1 << k;
    }
    if (!make_fill((const char*)fills + 16 * k, fill_bytes[k], a.fill[k])) return AREAL_ERR_BAD_ARG;
    a.src[k] = (const char*)src[k]; a.dst[k] = (char*)dst[k]; a.eb[k] = elem_bytes[k];
    max_eb = elem_bytes[k] > max_eb ? elem_bytes[k] : max_eb;
  }
  a.cu = cu_seqlens; a.cu_copy = cu_copy; a.cu_new = cu_new; a.n_seqs = (int)n_seqs; a.n_tensors = n_tensors;
  a.total = total; a.total_new = total_new; a.chunk = (int)pk_chunk_tokens(max_eb); a.host_total = host_total;
  const int64_t chunks = ceil_div_i64(total_new, a.chunk);
  if (chunks > PK_MAX_BLOCKS) return AREAL_ERR_UNSUPPORTED;
  hipLaunchKernelGGL(pad_packed_kernel, dim3((unsigned)chunks, (unsigned)(n_tensors > 0 ? n_tensors : 1)),
                     dim3(PK_THREADS), 0, stream, a);
  AREAL_CHECK_LAUNCH();
  return AREAL_OK;
}

size_t areal_masked_stats_workspace_bytes(int K) {
  if (K <= 0) return 0;
  return (size_t)K * STATS_BLOCKS * sizeof(StatPart) + 256;
}

// out [K][4] double = {sum, count, min, max} of values[k][i] over mask[k][i] != 0 (mask[k] NULL:
// every element). values / masks are HOST arrays of K device pointers, K <= 32.
int areal_masked_stats(const float* const* values, const uint8_t* const* masks, int K, int64_t n,
                       double* out, void* workspace, size_t workspace_bytes, hipStream_t stream) {
  if (K < 0 || K > STATS_MAX_K || n < 0) return AREAL_ERR_BAD_ARG;
  if (K == 0) return AREAL_OK;
  if (!values || !masks || !out) return AREAL_ERR_BAD_ARG;
  if (workspace == nullptr || workspace_bytes < areal_masked_stats_workspace_bytes(K))
    return AREAL_ERR_WORKSPACE;
  StatsArgs a;
  a.K = K; a.n = n;
  for (int k = 0; k < STATS_MAX_K; ++k) { a.v[k] = nullptr; a.m[k] = nullptr; }
  for (int k = 0; k < K; ++k) {
    if (values[k] == nullptr && n > 0) return AREAL_ERR_BAD_ARG;
    a.v[k] = values[k]; a.m[k] = masks[k];
  }
  StatPart* parts = (StatPart*)(((uintptr_t)workspace + 255) & ~(uintptr_t)255);
  int blocks = (int)ceil_div_i64(n > 0 ? n : 1, PK_THREADS * 8);
  if (blocks > STATS_BLOCKS) blocks = STATS_BLOCKS;
  if (blocks < 1) blocks = 1;
  hipLaunchKernelGGL(stats_partial_kernel, dim3(blocks, K), dim3(PK_THREADS), 0, stream, a, parts);
  AREAL_CHECK_LAUNCH();
  hipLaunchKernelGGL(stats_final_kernel, dim3(K), dim3(PK_THREADS), 0, stream, parts, blocks, out);
  AREAL_CHECK_LAUNCH();
  return AREAL_OK;
}

}  // extern "C"
