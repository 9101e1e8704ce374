// Packed-sequence GAE (segmented reverse scan) and masked group/batch normalisation.
//
// GAE follows areal/trainer/ppo/gae.py:10-36 (token-level recurrence on padded [bs, L]
// tensors); here it runs on the packed layout (or on the padded layout seen as bs sequences of
// length L). Normalisation follows areal/utils/data.py:1382-1637 (class Normalization) and
// areal/utils/functional/functional.py:16-53 (masked_normalization).
//
// GAE as a scan.  Going right to left, the carried state is (A, nv) = (last advantage, next
// value) and token t applies the affine map
//     A'  = A*((1-m) + c*m) + nv*(gamma*m) + (r - v)*m        c = gamma*lambda_seq
//     nv' = nv*(1-m) + v*m
// while the last token of a sequence applies the constant map (A', nv') = (0, no_eos ? v : 0).
// Affine maps compose associatively and constant maps absorb whatever lies to their right, so
// one unsegmented suffix scan over the whole packed array gives every sequence its own
// recurrence. Maps are held in fp64 (five coefficients); outputs are rounded to fp32.
#include <algorithm>
#include <atomic>
#include <chrono>
#include <random>

#include "common.hpp"

namespace {

// 16- and 8-byte accesses at any address of the element type
typedef f32x4 f32x4_any __attribute__((aligned(4)));
typedef u32x2 u32x2_any __attribute__((aligned(1)));

constexpr int GAE_THREADS = 256;
constexpr int GAE_ITEMS = 8;
constexpr int GAE_TILE = GAE_THREADS * GAE_ITEMS;
constexpr int GAE_SEG_WAVES = GAE_THREADS / 64;  // entries per (tile, group) segment of GaeArgs::seg_stats

// R = double in the three-launch scan (maps composed over the whole array); R = float in the
// single-pass kernel, where a map spans at most one tile and the state carried from tile to
// tile stays in fp64 (each output then sees ~20 fp32 roundings, like the reference's fp32 loop
// over as many tokens).
template <class R>
struct MapT {
  R a11, a12, a22, b1, b2;
};
using Map = MapT<double>;
using MapF = MapT<float>;
template <class R>
DEVI MapT<R> map_identity_t() { return MapT<R>{R(1), R(0), R(1), R(0), R(0)}; }
DEVI Map map_identity() { return map_identity_t<double>(); }
// (f o g): apply g first, then f.
template <class R>
DEVI MapT<R> compose(const MapT<R>& f, const MapT<R>& g) {
  // explicit fma: this file is compiled without contraction (the normalisation kernels follow
  // the reference's fp32 rounding), but the maps are more exact with it and cost half
  MapT<R> r;
  r.a11 = f.a11 * g.a11;
  r.a12 = fma(f.a11, g.a12, f.a12 * g.a22);
  r.a22 = f.a22 * g.a22;
  r.b1 = fma(f.a11, g.b1, fma(f.a12, g.b2, f.b1));
  r.b2 = fma(f.a22, g.b2, f.b2);
  return r;
}
// The map of the lane that CTRL names (common.hpp); the identity where that lane lies outside
// the row of 16.
template <int CTRL, class R>
DEVI MapT<R> dpp_map(const MapT<R>& m) {
  MapT<R> r;
  r.a11 = dpp_move<CTRL>(R(1), m.a11); r.a12 = dpp_move<CTRL>(R(0), m.a12);
  r.a22 = dpp_move<CTRL>(R(1), m.a22); r.b1 = dpp_move<CTRL>(R(0), m.b1);
  r.b2 = dpp_move<CTRL>(R(0), m.b2);
  return r;
}
template <class R>
DEVI MapT<R> lane_map(const MapT<R>& m, int lane) {
  return MapT<R>{lane_value(m.a11, lane), lane_value(m.a12, lane), lane_value(m.a22, lane),
                 lane_value(m.b1, lane), lane_value(m.b2, lane)};
}
// Inclusive suffix scan inside each row of 16 lanes: lane i gets the composition of the maps of
// lanes i..15 of its row (lane i applied last). No LDS traffic: the sixteen waves of a CU would
// queue at its one LDS unit with ds_bpermute shuffles.
template <class R>
DEVI MapT<R> row_suffix_scan(MapT<R> acc) {
  acc = compose(acc, dpp_map<DPP_ROW_SHL + 1>(acc));
  acc = compose(acc, dpp_map<DPP_ROW_SHL + 2>(acc));
  acc = compose(acc, dpp_map<DPP_ROW_SHL + 4>(acc));
  acc = compose(acc, dpp_map<DPP_ROW_SHL + 8>(acc));
  return acc;
}
// Composition of the maps of all 64 lanes (lane 0 applied last), in every lane.
template <class R>
DEVI MapT<R> wave_total_map(const MapT<R>& mine) {
  const MapT<R> acc = row_suffix_scan(mine);
  return compose(lane_map(acc, 0), compose(lane_map(acc, 16), compose(lane_map(acc, 32), lane_map(acc, 48))));
}
// Inclusive suffix scan over the wave: lane i gets the composition of lanes i..63.
template <class R>
DEVI MapT<R> wave_suffix_scan(const MapT<R>& mine, MapT<R>& total) {
  const MapT<R> acc = row_suffix_scan(mine);
  const MapT<R> t0 = lane_map(acc, 0), t1 = lane_map(acc, 16), t2 = lane_map(acc, 32), t3 = lane_map(acc, 48);
  const MapT<R> r1 = compose(t2, t3);  // all that lies right of row 1
  const MapT<R> r0 = compose(t1, r1);  // right of row 0
  total = compose(t0, r0);
  const int row = (threadIdx.x & 63) >> 4;
  const MapT<R> id = map_identity_t<R>();
  MapT<R> right;
  right.a11 = row == 0 ? r0.a11 : row == 1 ? r1.a11 : row == 2 ? t3.a11 : id.a11;
  right.a12 = row == 0 ? r0.a12 : row == 1 ? r1.a12 : row == 2 ? t3.a12 : id.a12;
  right.a22 = row == 0 ? r0.a22 : row == 1 ? r1.a22 : row == 2 ? t3.a22 : id.a22;
  right.b1 = row == 0 ? r0.b1 : row == 1 ? r1.b1 : row == 2 ? t3.b1 : id.b1;
  right.b2 = row == 0 ? r0.b2 : row == 1 ? r1.b2 : row == 2 ? t3.b2 : id.b2;
  return compose(acc, right);
}

// N sums at once: one pair of barriers instead of N.
template <int N>
DEVI void block_sum_n(double (&v)[N], double* smem /* [4][N] */) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
  for (int k = 0; k < N; ++k) v[k] = wave_sum(v[k]);
  __syncthreads();
  if (lane == 0) {
#pragma unroll
    for (int k = 0; k < N; ++k) smem[w * N + k] = v[k];
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < N; ++k) {
    double r = 0.0;
    for (int i = 0; i < (int)(blockDim.x >> 6); ++i) r += smem[i * N + k];
    v[k] = r;
  }
}

// ---- Sums handed from block to block inside a launch (adv_normalise_row, gae_tile_normalise): sealed words, N numbers
// and a check word made of them and the call's number, and a flag per entry, the call's number again, stored right behind
// them (a reader that sees the flag first finds the check word wrong and looks again; waiting for the words before storing
// it: packed GAE of 1.79 Mi tokens 27.1 -> 28.1 us). All go out and come in as agent-scope atomics (past the XCD's own L2); flags lie next to each other, so that
// looking again costs a line or two (with the words themselves looked at, 900 waiting blocks of 14 entries each slowed
// down the ones they waited for: packed GAE
// of 1.79 Mi tokens 31.4 -> 29.0 us). Whoever reads words that fit has
// all of them, whatever the memory held before (a chance of 2^-64 an entry otherwise), and nothing has to be cleared.
// Every word goes through a mix of its own (the multipliers of splitmix64): sums are doubles with few bits set (a count of 512 has one above its
// exponent's), and a sum of their products with odd numbers took entries for whole of which two counts were missing.
template <int N>
DEVI uint64_t sums_seal(uint64_t call, const uint64_t (&w)[N]) {
  uint64_t h = call;
#pragma unroll
  for (int k = 0; k < N; ++k) {
    h ^= w[k];
    h = (h ^ (h >> 32)) * 0xbf58476d1ce4e5b9ull;
    h = (h ^ (h >> 29)) * 0x94d049bb133111ebull;
  }
  return h ^ (h >> 32);
}
template <int N>
DEVI void publish_sums(uint64_t* to, uint64_t* flag, uint64_t call, const double (&s)[N]) {  // by one thread
  uint64_t w[N];
#pragma unroll
  for (int k = 0; k < N; ++k) {
    w[k] = __builtin_bit_cast(uint64_t, s[k]);
    __hip_atomic_store(to + k, w[k], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __hip_atomic_store(to + N, sums_seal(call, w), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __hip_atomic_store(flag, call, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// The sums of n entries PITCH words apart, added up by a whole wave: lane i takes every 64th from the i-th on, then the
// wave's sum. False when they were not all there at `deadline`.
template <int PITCH, int N>
DEVI bool gather_sums(const uint64_t* from, const uint64_t* flags, int n, uint64_t call, uint64_t deadline, double (&s)[N]) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int k = 0; k < N; ++k) s[k] = 0.0;
  for (int i = lane; i - lane < n; i += 64) {
    bool have = i >= n;
    for (;;) {
      if (!have && __hip_atomic_load(flags + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == call) {
        const uint64_t* const entry = from + (int64_t)PITCH * i;
        uint64_t w[N];
#pragma unroll
        for (int k = 0; k < N; ++k) w[k] = __hip_atomic_load(entry + k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const uint64_t seal = __hip_atomic_load(entry + N, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        have = seal == sums_seal(call, w);
        if (have) {
#pragma unroll
          for (int k = 0; k < N; ++k) s[k] += __builtin_bit_cast(double, w[k]);
        }
      }
      if (__builtin_amdgcn_ballot_w64(!have) == 0) break;
      if (wall_clock64() >= deadline) return false;
      __builtin_amdgcn_s_sleep(4);
    }
  }
#pragma unroll
  for (int k = 0; k < N; ++k) s[k] = wave_sum(s[k]);
  return true;
}
DEVI bool note_left(const uint64_t* left, uint64_t call) {
  return __hip_atomic_load(left, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == call;
}
// A block that leaves a note and looks at the sums again, and one that publishes its sums and looks for notes, each store
// to one address and load from another: both loads could be served ahead of both stores, each would miss the other, and
// the row or segment would stay without its normalisation. So a store and a fence come before the load on either side:
//   leaver      note       | fence               | flags of the sums, sums
//   publisher   sums, flag | wait for the stores | notes
// Whichever store is performed later, the load behind it sees the earlier one. The publisher's loads go past every cache
// that is not shared, so that waiting for the store is all of the fence it needs; store and load are of one wave on both
// sides. It costs nothing that shows: advantages of 64 x 1000 15.0 us, packed GAE of 1024 x 1750 27.1, both as without.
DEVI void leave_note(uint64_t* left, uint64_t call) {  // by one thread, whose wave looks again
  atomicExch((unsigned long long*)left, (unsigned long long)call);
  __threadfence();
}
DEVI void published_before_notes() { asm volatile("s_waitcnt vmcnt(0) ; flag out before notes are read" ::: "memory"); }
DEVI bool take_note(uint64_t* left, uint64_t call) {
  return atomicCAS((unsigned long long*)left, (unsigned long long)call, (unsigned long long)~call) == call;
}

struct GaeArgs {
  const float* rewards;
  const float* values;
  const float* mask;         // float 0/1
  const int32_t* cu;         // [n_seqs+1] or null when uniform_len > 0
  const uint8_t* no_eos;     // [n_seqs] or null (all false)
  const float* lam_seq;      // [n_seqs] per-sequence lambda or null
  int64_t n;
  int n_seqs;
  int64_t uniform_len;
  float discount;
  float lam;
  float* adv;
  float* ret;
  int block_per_seq;         // single-pass kernel, padded rows of at least a tile: block = row
  double* row_stats;         // nullable, with block_per_seq only: [5][n_seqs] sums over each row of
                             // m, x m, m^2, m^2 x, m^2 x^2 (x = the advantage written, m = mask):
                             // the statistics pass of the normalisation that follows, for free
  // packed tile kernel with statistics: the same five sums per (tile, group) segment. goff [G+1]
  // are the groups' token offsets (a partition of [0, n)); segment (tile k, group j) lands in slot
  // k + j of seg_stats [5][seg_slots][4] (one entry per wave of the tile's block), seg_slots =
  // tiles + G. Slots no segment maps to are zeroed.
  const int64_t* goff;
  int n_groups;
  double* seg_stats;
  int64_t seg_slots;
  const int64_t* gseq;       // the groups' first sequences [G+1] instead of their token offsets (goff null)
};
// Token offset of the first token of a group; as an array of the groups' ends from index 1 on.
struct GroupOffsets {
  const int64_t* goff;
  const int64_t* gseq;
  const int32_t* cu;
  int shift;
  DEVI int64_t operator[](int j) const { return goff != nullptr ? goff[j + shift] : (int64_t)cu[gseq[j + shift]]; }
};
DEVI GroupOffsets group_offsets(const GaeArgs& g, int shift = 0) { return GroupOffsets{g.goff, g.gseq, g.cu, shift}; }

DEVI int gae_seq_of(const GaeArgs& g, int64_t t) {
  if (g.uniform_len > 0) return (int)(t / g.uniform_len);
  int lo = 0, hi = g.n_seqs;
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if ((int64_t)g.cu[mid] <= t) lo = mid; else hi = mid;
  }
  return lo;
}
DEVI int64_t gae_seq_end(const GaeArgs& g, int s) {
  return g.uniform_len > 0 ? (int64_t)(s + 1) * g.uniform_len : (int64_t)g.cu[s + 1];
}

// Maps of the thread's GAE_ITEMS consecutive tokens starting at t0 (identity beyond n).
DEVI void load_maps(const GaeArgs& g, int64_t t0, Map (&mp)[GAE_ITEMS], float (&v)[GAE_ITEMS]) {
  if (t0 >= g.n) {
#pragma unroll
    for (int i = 0; i < GAE_ITEMS; ++i) { mp[i] = map_identity(); v[i] = 0.f; }
    return;
  }
  float rw[GAE_ITEMS], ms[GAE_ITEMS];
  if (t0 + GAE_ITEMS <= g.n) {  // t0 is a multiple of GAE_ITEMS: 16-byte aligned vector loads
#pragma unroll
    for (int q = 0; q < GAE_ITEMS / 4; ++q) {
      const f32x4 a = *(const f32x4*)(g.rewards + t0 + 4 * q);
      const f32x4 b = *(const f32x4*)(g.values + t0 + 4 * q);
      const f32x4 c = *(const f32x4*)(g.mask + t0 + 4 * q);
#pragma unroll
      for (int e = 0; e < 4; ++e) { rw[4 * q + e] = a[e]; v[4 * q + e] = b[e]; ms[4 * q + e] = c[e]; }
    }
  } else {
#pragma unroll
    for (int i = 0; i < GAE_ITEMS; ++i) {
      const bool in = t0 + i < g.n;
      rw[i] = in ? g.rewards[t0 + i] : 0.f;
      v[i] = in ? g.values[t0 + i] : 0.f;
      ms[i] = in ? g.mask[t0 + i] : 0.f;
    }
  }
  int s = gae_seq_of(g, t0);
  int64_t e = gae_seq_end(g, s);
#pragma unroll
  for (int i = 0; i < GAE_ITEMS; ++i) {
    const int64_t t = t0 + i;
    if (t >= g.n) { mp[i] = map_identity(); v[i] = 0.f; continue; }
    while (t >= e && s + 1 < g.n_seqs) { ++s; e = gae_seq_end(g, s); }
    const float val = v[i];
    if (t == e - 1) {
      const bool ne = g.no_eos != nullptr && g.no_eos[s] != 0;
      mp[i] = Map{0.0, 0.0, 0.0, 0.0, ne ? (double)val : 0.0};
    } else {
      const double m = (double)ms[i];
      const double lam = g.lam_seq != nullptr ? (double)g.lam_seq[s] : (double)g.lam;
      const double c = (double)g.discount * lam;
      Map f;
      f.a11 = (1.0 - m) + c * m;
      f.a12 = (double)g.discount * m;
      f.a22 = 1.0 - m;
      f.b1 = ((double)rw[i] - (double)val) * m;
      f.b2 = (double)val * m;
      mp[i] = f;
    }
  }
}

// Composition of the thread's maps: leftmost applied last.
DEVI Map thread_total(const Map (&mp)[GAE_ITEMS]) {
  Map r = mp[GAE_ITEMS - 1];
#pragma unroll
  for (int i = GAE_ITEMS - 2; i >= 0; --i) r = compose(mp[i], r);
  return r;
}

// Inclusive suffix scan over the block: returns for each thread the composition of the maps
// of threads tid..blockDim-1 (thread tid applied last). smem: one slot per wave.
template <class R>
DEVI MapT<R> block_suffix_scan(MapT<R> mine, MapT<R>* smem, MapT<R>& block_total) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  MapT<R> wave_total;
  const MapT<R> acc = wave_suffix_scan(mine, wave_total);
  __syncthreads();
  if (lane == 0) smem[w] = wave_total;
  __syncthreads();
  const int nw = blockDim.x >> 6;
  MapT<R> right = map_identity_t<R>();
  for (int i = nw - 1; i > w; --i) right = compose(smem[i], right);
  MapT<R> tot = right;
  for (int i = w; i >= 0; --i) tot = compose(smem[i], tot);
  block_total = tot;
  return compose(acc, right);
}

__global__ __launch_bounds__(GAE_THREADS) void gae_block_total_kernel(GaeArgs g, Map* totals) {
  __shared__ Map smem[4];
  const int64_t t0 = (int64_t)blockIdx.x * GAE_TILE + (int64_t)threadIdx.x * GAE_ITEMS;
  Map mp[GAE_ITEMS];
  float v[GAE_ITEMS];
  load_maps(g, t0, mp, v);
  Map total;
  block_suffix_scan(thread_total(mp), smem, total);
  if (threadIdx.x == 0) totals[blockIdx.x] = total;
}

// carry[b] = state (A, nv) entering block b from its right = (F_{b+1} o F_{b+2} o ...)(0, 0).
__global__ __launch_bounds__(GAE_THREADS) void gae_carry_kernel(const Map* totals, int nblocks,
                                                                double* carry) {
  __shared__ Map smem[4];
  const int per = (nblocks + GAE_THREADS - 1) / GAE_THREADS;
  const int b0 = threadIdx.x * per;
  // composition of this thread's blocks b0 .. b0+per-1
  Map mine = map_identity();
  for (int i = per - 1; i >= 0; --i) {
    const int b = b0 + i;
    if (b < nblocks) mine = compose(totals[b], mine);
  }
  Map total;
  const Map incl = block_suffix_scan(mine, smem, total);
  // exclusive: composition of everything right of this thread's range
  Map excl;
  {
    // incl = mine o right  =>  right is what enters after this thread's range; recompute it
    // from the neighbour: thread tid+1's inclusive scan equals our exclusive one.
    __shared__ Map all[GAE_THREADS];
    all[threadIdx.x] = incl;
    __syncthreads();
    excl = threadIdx.x + 1 < blockDim.x ? all[threadIdx.x + 1] : map_identity();
  }
  // walk this thread's blocks right to left
  double A = excl.b1, nv = excl.b2;  // map applied to the zero state
  for (int i = per - 1; i >= 0; --i) {
    const int b = b0 + i;
    if (b >= nblocks) continue;
    carry[2 * b] = A;
    carry[2 * b + 1] = nv;
    const Map f = totals[b];
    const double A2 = fma(f.a11, A, fma(f.a12, nv, f.b1));
    const double nv2 = fma(f.a22, nv, f.b2);
    A = A2; nv = nv2;
  }
}

__global__ __launch_bounds__(GAE_THREADS) void gae_apply_kernel(GaeArgs g, const double* carry) {
  __shared__ Map smem[4];
  __shared__ Map all[GAE_THREADS];
  const int64_t t0 = (int64_t)blockIdx.x * GAE_TILE + (int64_t)threadIdx.x * GAE_ITEMS;
  Map mp[GAE_ITEMS];
  float v[GAE_ITEMS];
  load_maps(g, t0, mp, v);
  Map total;
  const Map incl = block_suffix_scan(thread_total(mp), smem, total);
  all[threadIdx.x] = incl;
  __syncthreads();
  const Map excl = threadIdx.x + 1 < blockDim.x ? all[threadIdx.x + 1] : map_identity();
  const double A0 = carry[2 * blockIdx.x], nv0 = carry[2 * blockIdx.x + 1];
  double A = excl.a11 * A0 + excl.a12 * nv0 + excl.b1;
  double nv = excl.a22 * nv0 + excl.b2;
#pragma unroll
  for (int i = GAE_ITEMS - 1; i >= 0; --i) {
    const int64_t t = t0 + i;
    if (t >= g.n) continue;
    const Map& f = mp[i];
    const double A2 = fma(f.a11, A, fma(f.a12, nv, f.b1));
    const double nv2 = fma(f.a22, nv, f.b2);
    A = A2; nv = nv2;
    const float a = (float)A;
    g.adv[t] = a;
    g.ret[t] = a + v[i];
  }
}

// ---------------------------------------------------------------------------------------
// Single-pass GAE: one launch, every token read once and written once (20 B/token), no block
// has to wait for another. Sequences are independent, so nothing enters a sequence's last token from
// its right. Two kernels:
//  * padded rows (gae_owned_kernel): block b owns the rows whose END lies in the token range
//    (b*TILE, (b+1)*TILE] (one block per row when rows are at least a tile long) and walks them
//    right to left tile by tile, carrying (A, nv) across its tiles;
//  * packed sequences (gae_tile_kernel): block = tile; the state entering the tile is made from the maps of the
//    crossing sequence's remaining tokens, recomputed or, where the launch hands them over, those of their blocks.
// Tiles are absolute multiples of TILE, so the 16-byte loads stay aligned. The host picks the
// three-launch scan above when sequences are long on average.
// ---------------------------------------------------------------------------------------

// One tile of the single-pass kernels: the block's 256 threads take 8 consecutive tokens each
// of tile `tile` (tokens [tile * TILE, (tile + 1) * TILE)), of which [t_begin, t_end) are this
// block's to write. cu_own[i] = cu[s_first + i] for i in [0, n_own] covers every sequence that
// holds one of those tokens (cu_own[0] <= t_begin, cu_own[n_own] >= t_end); with uniform rows
// cu_own is unused. (A0, nv0) is the fp64 state entering the tile from its right and is replaced
// by the state leaving it on the left.
// oa receives the advantages of the thread's owned tokens (zero elsewhere).
// The thread's 8 consecutive tokens from t0 (a multiple of 8) as raw inputs; zeros where `want`
// is false and beyond the array. Without values (no critic) they are zero too.
DEVI void gae_load_items(const GaeArgs& g, int64_t t0, bool want, float (&rw)[GAE_ITEMS],
                         float (&v)[GAE_ITEMS], float (&ms)[GAE_ITEMS]) {
#pragma unroll
  for (int i = 0; i < GAE_ITEMS; ++i) { rw[i] = 0.f; v[i] = 0.f; ms[i] = 0.f; }
  if (!want) return;
  if (t0 + GAE_ITEMS <= g.n) {
#pragma unroll
    for (int q = 0; q < GAE_ITEMS / 4; ++q) {
      const f32x4 a = *(const f32x4*)(g.rewards + t0 + 4 * q);
      f32x4 b = {0.f, 0.f, 0.f, 0.f};
      if (g.values != nullptr) b = *(const f32x4*)(g.values + t0 + 4 * q);
      const f32x4 c = *(const f32x4*)(g.mask + t0 + 4 * q);
#pragma unroll
      for (int e = 0; e < 4; ++e) { rw[4 * q + e] = a[e]; v[4 * q + e] = b[e]; ms[4 * q + e] = c[e]; }
    }
  } else {
#pragma unroll
    for (int i = 0; i < GAE_ITEMS; ++i) {
      const bool in = t0 + i < g.n;
      rw[i] = in ? g.rewards[t0 + i] : 0.f;
      v[i] = in && g.values != nullptr ? g.values[t0 + i] : 0.f;
      ms[i] = in ? g.mask[t0 + i] : 0.f;
    }
  }
}

// local indices [i_lo, i_hi) of the thread's 8 tokens from t0 that lie in [t_begin, t_end)
DEVI void gae_owned_items(int64_t t0, int64_t t_begin, int64_t t_end, int& i_lo, int& i_hi) {
  const int64_t d_lo = t_begin - t0, d_hi = t_end - t0;
  i_lo = d_lo > 0 ? (d_lo < GAE_ITEMS ? (int)d_lo : GAE_ITEMS) : 0;
  i_hi = d_hi < GAE_ITEMS ? (d_hi > 0 ? (int)d_hi : 0) : GAE_ITEMS;
}

// How a tile finds its sequences: in cu_seqlens, or as rows of uniform length.
enum { GAE_LAYOUT_CU = 0, GAE_LAYOUT_ROWS = 1 };

// (rw, v, ms): the tile's inputs as gae_load_items leaves them (at least the owned tokens).
// LAMBDAS: a lambda per sequence (GaeArgs::lam_seq).
template <int LAYOUT, bool LAMBDAS>
DEVI void gae_one_tile(const GaeArgs& g, int64_t tile, int64_t t_begin, int64_t t_end, int s_first,
                       int n_own, const int32_t* cu_own, double& A0, double& nv0,
                       MapF* smem, MapF* all,
                       const float (&rw)[GAE_ITEMS], const float (&v)[GAE_ITEMS],
                       const float (&ms)[GAE_ITEMS], float (&oa)[GAE_ITEMS]) {
  constexpr bool uniform = LAYOUT != GAE_LAYOUT_CU;
  const int tid = threadIdx.x;
  const int64_t t0 = tile * GAE_TILE + (int64_t)tid * GAE_ITEMS;
  // The thread keeps its 8 tokens as raw inputs plus two bit masks and rebuilds a token's map
  // where it is needed (twice): holding 8 maps would cost a wave of occupancy.
  float lm[LAMBDAS ? GAE_ITEMS : 1], mm[GAE_ITEMS];
  unsigned valid = 0, ends = 0, boot = 0;  // bit i: token owned / last of its sequence / no_eos
  int i_lo, i_hi;  // owned tokens of this thread
  gae_owned_items(t0, t_begin, t_end, i_lo, i_hi);
  const bool any = i_lo < i_hi;
  if (LAMBDAS) {
#pragma unroll
    for (int i = 0; i < (LAMBDAS ? GAE_ITEMS : 1); ++i) lm[i] = g.lam;
  }
  if (any) {
    // sequence of the first owned token of this thread (index relative to s_first)
    const int64_t tf = t0 + i_lo;
    int sq;
    int e_loc;  // local index one past the last token of sequence sq (clamped)
    if (LAYOUT == GAE_LAYOUT_ROWS) {
      sq = (int)(tf / g.uniform_len) - s_first;
      const int64_t e = (int64_t)(sq + s_first + 1) * g.uniform_len - t0;
      e_loc = e < 2 * GAE_ITEMS ? (int)e : 2 * GAE_ITEMS;
    } else {
      int a = 0, b = n_own;  // cu_own[a] <= tf < cu_own[b]
      while (b - a > 1) {
        const int mid = (a + b) >> 1;
        if ((int64_t)cu_own[mid] <= tf) a = mid; else b = mid;
      }
      sq = a;
      const int64_t e = (int64_t)cu_own[sq + 1] - t0;
      e_loc = e < 2 * GAE_ITEMS ? (int)e : 2 * GAE_ITEMS;
    }
    valid = ((1u << i_hi) - 1u) & ~((1u << i_lo) - 1u);
    if (e_loc > i_hi && !LAMBDAS) {
      // common case: all owned tokens inside one sequence, none of them its last
    } else {
      // a sequence ends among these tokens (or lambda is per sequence): walk them
      for (int i = i_lo; i < i_hi; ++i) {
        while (i >= e_loc && sq + 1 < n_own) {
          ++sq;
          const int64_t e = (uniform ? (int64_t)(sq + s_first + 1) * g.uniform_len
                                     : (int64_t)cu_own[sq + 1]) - t0;
          e_loc = e < 2 * GAE_ITEMS ? (int)e : 2 * GAE_ITEMS;
        }
        if (LAMBDAS) {
          const float l = g.lam_seq[s_first + sq];
#pragma unroll
          for (int k = 0; k < (LAMBDAS ? GAE_ITEMS : 1); ++k) if (k == i) lm[k] = l;
        }
        if (i == e_loc - 1) {
          ends |= 1u << i;
          if (g.no_eos != nullptr && g.no_eos[s_first + sq] != 0) boot |= 1u << i;
        }
      }
    }
  }
  // not owned: identity (mask 0 with no offsets)
#pragma unroll
  for (int i = 0; i < GAE_ITEMS; ++i) mm[i] = ((valid >> i) & 1u) ? ms[i] : 0.f;
  const float gam = g.discount;
  const float c0 = gam * g.lam;
  // few waves hold the last token of a sequence: the others skip its constant map by a scalar branch
  const bool wave_has_end = __builtin_amdgcn_ballot_w64(ends != 0) != 0;
  auto token_map = [&](int i) -> MapF {
    const float val = v[i];
    const float m = mm[i];
    const float c = LAMBDAS ? gam * lm[LAMBDAS ? i : 0] : c0;
    MapF f;
    f.a11 = fmaf(c, m, 1.f - m);
    f.a12 = gam * m;
    f.a22 = 1.f - m;
    f.b1 = (rw[i] - val) * m;
    f.b2 = val * m;
    if (wave_has_end) {
      if ((ends >> i) & 1u) f = MapF{0.f, 0.f, 0.f, 0.f, ((boot >> i) & 1u) ? val : 0.f};
    }
    return f;
  };
  MapF mine = token_map(GAE_ITEMS - 1);
#pragma unroll
  for (int i = GAE_ITEMS - 2; i >= 0; --i) mine = compose(token_map(i), mine);
  MapF total;
  const MapF incl = block_suffix_scan(mine, smem, total);
  all[tid] = incl;
  __syncthreads();
  const MapF excl = tid + 1 < GAE_THREADS ? all[tid + 1] : map_identity_t<float>();
  // the state entering this thread's tokens: the fp32 map of everything to its right in the
  // tile applied to the fp64 state entering the tile
  float A = (float)fma((double)excl.a11, A0, fma((double)excl.a12, nv0, (double)excl.b1));
  float nv = (float)fma((double)excl.a22, nv0, (double)excl.b2);
#pragma unroll
  for (int i = 0; i < GAE_ITEMS; ++i) oa[i] = 0.f;
  if (any) {
    float orr[GAE_ITEMS];
#pragma unroll
    for (int i = GAE_ITEMS - 1; i >= 0; --i) {
      const MapF f = token_map(i);
      const float A2 = fmaf(f.a11, A, fmaf(f.a12, nv, f.b1));
      const float nv2 = fmaf(f.a22, nv, f.b2);
      A = A2; nv = nv2;
      oa[i] = A;
      orr[i] = oa[i] + v[i];
    }
    if (valid == (1u << GAE_ITEMS) - 1u) {
#pragma unroll
      for (int q = 0; q < GAE_ITEMS / 4; ++q) {
        *(f32x4_any*)(g.adv + t0 + 4 * q) = f32x4{oa[4 * q], oa[4 * q + 1], oa[4 * q + 2], oa[4 * q + 3]};
        *(f32x4_any*)(g.ret + t0 + 4 * q) = f32x4{orr[4 * q], orr[4 * q + 1], orr[4 * q + 2], orr[4 * q + 3]};
      }
    } else {
#pragma unroll
      for (int i = 0; i < GAE_ITEMS; ++i)
        if ((valid >> i) & 1u) { g.adv[t0 + i] = oa[i]; g.ret[t0 + i] = orr[i]; }
    }
  }
  // state entering the next tile on the left
  const double A1 = fma((double)total.a11, A0, fma((double)total.a12, nv0, (double)total.b1));
  const double nv1 = fma((double)total.a22, nv0, (double)total.b2);
  A0 = A1; nv0 = nv1;
}

// ---------------------------------------------------------------------------------------
// One row walked by one block (gae_owned_kernel<ONE_ROW>, adv_gae_kernel), tile by tile of the row from the right. A
// thread has two quads of 4 tokens a tile, WAVE_QUADS tokens apart, so that every access of a wave is 1 KiB in one
// piece; the maps of the two quads are scanned side by side. With 8 tokens in a row to a thread, each of its 16-byte
// stores left every other 16 bytes of a line to the next instruction: adv_gae_kernel with inputs new to the caches, at
// 1024 x 8192 with critic and reference, 81 us, in quads 70; at 1000 x 8191 without a critic 78 and 67.
// ---------------------------------------------------------------------------------------
constexpr int QUAD = 4, WAVE_QUADS = 64 * QUAD;  // tokens of one 16-byte access of a thread / of a wave
constexpr int ROW_QUADS = GAE_ITEMS / QUAD;
typedef MapF RowMaps[2][GAE_THREADS / 64];  // of the waves, in LDS, alternating from tile to tile

// Row token of the calling thread's first quad.
DEVI int row_tile_token(int tile) {
  const int tid = threadIdx.x;
  return tile * GAE_TILE + (tid >> 6) * ROW_QUADS * WAVE_QUADS + (tid & 63) * QUAD;
}

// Quad q of the thread's tokens from t0 on of a row of L tokens. STREAM: non-temporal, which pays for some of
// adv_gae_kernel's arrays (log-probs and KL rewards: 70 -> 66 and 67 -> 60 us in the cases above) and for all of
// them does not (73 and 75).
template <bool STREAM>
DEVI void row_store(float* to, int t0, int L, int q, const f32x4& w) {
  const int tq = t0 + q * WAVE_QUADS;
  if (tq + QUAD <= L) {
    if constexpr (STREAM) __builtin_nontemporal_store(w, (f32x4_any*)(to + tq));
    else *(f32x4_any*)(to + tq) = w;
  } else {
#pragma unroll
    for (int e = 0; e < QUAD - 1; ++e)
      if (tq + e < L) to[tq + e] = w[e];
  }
}

// The mask of a thread's tokens as bytes (nonzero = 1) or floats. again(): what was worked out from it before is not
// held in registers beyond this point.
struct ByteMask {
  uint32_t (&m)[ROW_QUADS];
  DEVI float operator()(int i) const { return (m[i / QUAD] >> (8 * (i % QUAD))) & 0xffu ? 1.f : 0.f; }
  DEVI void again() const {
#pragma unroll
    for (int q = 0; q < ROW_QUADS; ++q) asm volatile("" : "+v"(m[q]));
  }
};
struct FloatMask {
  const float (&m)[GAE_ITEMS];
  DEVI float operator()(int i) const { return m[i]; }
  DEVI void again() const {}
};

// rw, v: rewards and values of the thread's tokens (zero beyond the row). mask_of(i): their mask, zero beyond the row
// (which makes such a token the identity). boot: whether the row's last value is bootstrapped. (A0, nv0): the fp64 state entering the tile from its
// right, replaced by the one leaving it on the left. rs: the row's sums of GaeArgs::row_stats (STATS). put_adv(q, x): takes
// the advantages of quad q. ret: the row.
template <bool STATS, bool BINARY, class Mask, class PutAdv>
DEVI void gae_row_tile(float gam, float lam, int tile, int t0, int L, bool boot, float (&rw)[GAE_ITEMS],
                       float (&v)[GAE_ITEMS], const Mask& mask_of, RowMaps& maps, double& A0, double& nv0,
                       double (&rs)[STATS ? 5 : 1], const PutAdv& put_adv, float* ret) {
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const float c0 = gam * lam;
  const int last = L - 1 - t0;
  const bool wave_has_end = __builtin_amdgcn_ballot_w64(last >= 0 && last < WAVE_QUADS + QUAD) != 0;
  auto token_map = [&](int i) -> MapF {
    const float m = mask_of(i);
    MapF f;
    f.a11 = fmaf(c0, m, 1.f - m);
    f.a12 = gam * m;
    f.a22 = 1.f - m;
    f.b1 = (rw[i] - v[i]) * m;
    f.b2 = v[i] * m;
    if (wave_has_end) {
      if (last == (i / QUAD) * WAVE_QUADS + i % QUAD) f = MapF{0.f, 0.f, 0.f, 0.f, boot ? v[i] : 0.f};
    }
    return f;
  };
  MapF incl[ROW_QUADS], total[ROW_QUADS];
#pragma unroll
  for (int q = 0; q < ROW_QUADS; ++q) {
    MapF mine = token_map(QUAD * q + QUAD - 1);
#pragma unroll
    for (int e = QUAD - 2; e >= 0; --e) mine = compose(token_map(QUAD * q + e), mine);
    incl[q] = wave_suffix_scan(mine, total[q]);
  }
  MapF* const waves = maps[tile & 1];  // (the other half's readers are past the barrier behind it)
  if (lane == 0) waves[wave] = compose(total[0], total[1]);
  __syncthreads();
  auto advance = [](const MapF& f, double& A, double& nv) {
    const double A1 = fma((double)f.a11, A, fma((double)f.a12, nv, (double)f.b1));
    nv = fma((double)f.a22, nv, (double)f.b2);
    A = A1;
  };
  double Aw = A0, nw = nv0;  // the state entering the wave's tokens
#pragma unroll
  for (int w = GAE_THREADS / 64 - 1; w >= 0; --w) {
    if (w == wave) { Aw = A0; nw = nv0; }
    advance(waves[w], A0, nv0);
  }
  // (the token maps are worked out again rather than held: 40 registers)
#pragma unroll
  for (int i = 0; i < GAE_ITEMS; ++i) asm volatile("" : "+v"(rw[i]), "+v"(v[i]));
  mask_of.again();
#pragma unroll
  for (int q = ROW_QUADS - 1; q >= 0; --q) {
    const MapF id = map_identity_t<float>();
    const MapF excl = {wave_shift_down(incl[q].a11, id.a11), wave_shift_down(incl[q].a12, id.a12),
                       wave_shift_down(incl[q].a22, id.a22), wave_shift_down(incl[q].b1, id.b1),
                       wave_shift_down(incl[q].b2, id.b2)};
    double At = Aw, nt = nw;
    advance(excl, At, nt);
    float A = (float)At, nv = (float)nt;
    f32x4 o_adv, o_ret;
#pragma unroll
    for (int e = QUAD - 1; e >= 0; --e) {
      const int i = QUAD * q + e;
      const MapF f = token_map(i);
      const float A2 = fmaf(f.a11, A, fmaf(f.a12, nv, f.b1));
      nv = fmaf(f.a22, nv, f.b2);
      A = A2;
      o_adv[e] = A;
      o_ret[e] = A + v[i];
      if constexpr (STATS) {
        const float m = mask_of(i);
        if (m != 0.f) {
          const double x = (double)A;
          if (BINARY || m == 1.f) {  // the usual 0/1 mask: one fp64 multiplication per token
            rs[0] += 1.0; rs[1] += x; rs[4] += x * x;
            if (!BINARY) { rs[2] += 1.0; rs[3] += x; }
          } else {
            const double md = (double)m;
            const double xm = x * md, mm = md * md;
            rs[0] += md; rs[1] += xm; rs[2] += mm; rs[3] += xm * md; rs[4] += xm * xm;
          }
        }
      }
    }
    put_adv(q, o_adv);
    row_store<false>(ret, t0, L, q, o_ret);
    advance(total[q], Aw, nw);
  }
}

// (Blocks of 1024 threads, one 8192-token tile per padded row instead of four serial tiles of
// 2048, measured slower: 46.7 against 30.8 us on [1024, 8192]; one such block fills a CU's
// registers and the latency of its single pass is not covered by anything.)
// STATS: also sum each row's advantages under the mask (block = row only), see GaeArgs::row_stats.
// ONE_ROW: block = row (GaeArgs::block_per_seq); LAMBDAS: a lambda per row.
template <bool STATS, bool ONE_ROW, bool LAMBDAS>
__global__ __launch_bounds__(GAE_THREADS, 4) void gae_owned_kernel(GaeArgs g) {
  if constexpr (ONE_ROW) {
    __shared__ RowMaps maps;
    const int b = blockIdx.x, L = (int)g.uniform_len;
    const int64_t row = (int64_t)b * L;
    const float lam = LAMBDAS ? g.lam_seq[b] : g.lam;
    const bool boot = g.no_eos != nullptr && g.no_eos[b] != 0;
    double A0 = 0.0, nv0 = 0.0;  // state entering the current tile from its right
    double rs[STATS ? 5 : 1] = {0.0};
    for (int tile = (L - 1) / GAE_TILE; tile >= 0; --tile) {
      const int t0 = row_tile_token(tile);
      float rw[GAE_ITEMS], v[GAE_ITEMS], ms[GAE_ITEMS];
      auto load = [&](const float* from, float (&x)[GAE_ITEMS]) {
#pragma unroll
        for (int i = 0; i < GAE_ITEMS; ++i) x[i] = 0.f;
        if (from == nullptr) return;
#pragma unroll
        for (int q = 0; q < ROW_QUADS; ++q) {
          const int tq = t0 + q * WAVE_QUADS;
          if (tq + QUAD <= L) {
            const f32x4 w = *(const f32x4_any*)(from + row + tq);
#pragma unroll
            for (int e = 0; e < QUAD; ++e) x[QUAD * q + e] = w[e];
          } else {
#pragma unroll
            for (int e = 0; e < QUAD; ++e)
              if (tq + e < L) x[QUAD * q + e] = from[row + tq + e];
          }
        }
      };
      load(g.rewards, rw);
      load(g.values, v);
      load(g.mask, ms);
      gae_row_tile<STATS, false>(
          g.discount, lam, tile, t0, L, boot, rw, v, FloatMask{ms}, maps, A0, nv0, rs,
          [&](int q, const f32x4& w) { row_store<false>(g.adv + row, t0, L, q, w); }, g.ret + row);
    }
    if constexpr (STATS) {
      __shared__ double s_rs[4 * 5];
      block_sum_n<5>(rs, s_rs);
      if (threadIdx.x == 0) {
#pragma unroll
        for (int k = 0; k < 5; ++k) g.row_stats[(int64_t)k * g.n_seqs + b] = rs[k];
      }
    }
    return;
  }
  __shared__ MapF smem[GAE_THREADS / 64];
  __shared__ MapF all[GAE_THREADS];
  const int tid = threadIdx.x;
  // Workgroups go to the 8 XCDs round-robin by id. Giving XCD x the x-th eighth of the token
  // ranges keeps neighbouring ranges on one XCD.
  const int64_t per_xcd = (gridDim.x + 7) >> 3;
  const int64_t range = (int64_t)(blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
  const int64_t lo = range * GAE_TILE;
  if (range >= per_xcd * 8 || lo >= g.n) return;
  const int64_t hi = lo + GAE_TILE < g.n ? lo + GAE_TILE : g.n;
  // owned rows [s_first, s_last]: lo < end(s) <= hi
  const int s_first = (int)(lo / g.uniform_len);
  const int s_last = (int)(hi / g.uniform_len) - 1;
  if (s_first > s_last) return;  // uniform for the block
  const int n_own = s_last - s_first + 1;
  const int64_t t_begin = (int64_t)s_first * g.uniform_len;
  const int64_t t_end = (int64_t)(s_last + 1) * g.uniform_len;

  double A0 = 0.0, nv0 = 0.0;  // state entering the current tile from its right
  for (int64_t tile = (t_end - 1) / GAE_TILE; tile >= t_begin / GAE_TILE; --tile) {
    const int64_t t0 = tile * GAE_TILE + (int64_t)tid * GAE_ITEMS;
    int i_lo, i_hi;
    gae_owned_items(t0, t_begin, t_end, i_lo, i_hi);
    float rw[GAE_ITEMS], v[GAE_ITEMS], ms[GAE_ITEMS], oa[GAE_ITEMS];
    gae_load_items(g, t0, i_lo < i_hi, rw, v, ms);
    gae_one_tile<GAE_LAYOUT_ROWS, LAMBDAS>(g, tile, t_begin, t_end, s_first, n_own, nullptr, A0, nv0, smem, all, rw, v,
                                           ms, oa);
  }
}

// Single-pass GAE for packed sequences of ordinary length, one block per tile. What enters the
// tile from its right is the state of the sequence that crosses the tile's right edge, and it
// depends only on that sequence's tokens beyond the edge: maps of chunks of 512 tokens, a wave each, applied to the zero
// state in fp64 from the right. Those of the tile with its last token the block makes itself (rewards, values, mask are read,
// nothing written, the next chunk on its way while one is composed; a wave whose chunk holds none of it reads nothing). Those
// of whole tiles between are the totals that these tiles' blocks need anyway: the launch that normalises hands them
// over (TileMaps), 16 tiles at a time, for otherwise a sequence of k tiles is read k / 2 times, one chunk after the other;
// where they do not come in time, and in gae_tile_kernel, which has no words for them, the block makes them too: the same
// numbers, so the same bits. One launch, us, with the code that made them all in each block / so, lognormal lengths of deviation 0.8:
// 1024 x 1750 26.4 / 25.1 (29.4 / 28.7 with inputs new to the caches), 512 x 4000 35.7 / 27.1, 64 x 8192 41.0 / 18.8, 256 x 1750 19.1 /
// 15.9; of deviation 1.5, 512 x 3000 57.2 / 29.1; 0.5, 32 x 16000 31.6 / 19.1; equal lengths, which cross two whole tiles at most,
// 64 x 8192 15.1 / 15.3, 128 x 8192 19.3 / 19.1 (new inputs 21.5 / 21.9). Two launches, where each block still makes them, chunk by
// chunk: 64 x 8192 42.6 / 40.1, 512 x 3000 58.7 / 55.1, 512 x 8192 of equal lengths 52.8 / 48.3. Handing over maps of a sequence over one
// or two whole tiles too pays (1024 x 1600 25.2; from 2 tiles on 26.4, from 3 27.4).
// Against blocks that walk the sequences they own tile by tile, carrying the state (the padded-row kernel above, which
// also took cu_seqlens once): faster on 64 x 16384 tokens and on 4 x 32768, where a walking block has 16 tiles in a row.
// The layout comes first. Up to 2048 sequences (and 1024 groups) cu_seqlens and the groups' first sequences go to LDS
// whole, and what the tile has to find in them is counted from the registers on the way: one barrier, no load that waits
// for another. Above 2048 a wave searches for the sequences: its first 64 probes go out with the block's first loads, one more
// load of 128 entries holds all that the tile needs of up to 4096 sequences, and the groups are counted in LDS from what it
// finds. With 4096 in LDS (16 loads a thread) 4000 sequences of 300 took 21.3 us, with this search 20.7; with searches by all
// waves that wait for each other (of groups, first and last sequence, then their starts) 4096 x 300 took 20.2, with this one 20.6, 4096 x
// 1000 in eights 54.0 and 51.8.
// The kernel is bound by vector instruction issue (about 1150 vector and 250 scalar instructions
// per wave and tile on 1024 sequences of mean length 1760, half as many again with the group sums) for half of its time and by
// the chain of loads, maps and sums for the other half, with four blocks resident per CU, so
// that all blocks of a 1.8 M-token batch run at once; that leaves 128 registers.
constexpr int GAE_CHUNK = 64 * GAE_ITEMS;  // tokens of a wave's step through the crossing sequence
constexpr int GAE_CU_LDS = 8 * GAE_THREADS;  // sequences whose starts the block can hold (>= TILE + 1)
constexpr int GAE_GROUPS_LDS = 4 * GAE_THREADS;  // groups whose first sequences it can hold

// Groups of a tile for GaeArgs::seg_stats: those of the tile's first and last token and of the next
// tile's first token, each the number of group ends at or before the token. Waves 0..2 search
// (their loads go out with the tile's own); s_grp is valid after the block's next barrier.
DEVI void gae_tile_group_search(const GaeArgs& g, int64_t lo, int64_t hi, int* s_grp /* [3] */) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (wave < 3) {
    const int64_t x = wave == 0 ? lo : (wave == 1 ? hi - 1 : hi);
    const int r = wave_count_le(group_offsets(g, 1), g.n_groups, x, lane);
    if (lane == 0) s_grp[wave] = r;
  }
}

// Group bounds of a tile relative to its first token, kept in registers from the start of the
// kernel to its end: b[i] = goff[g_first + i] - lo for the first three bounds.
struct GaeTileGroups {
  int g_first, g_last, g_next;
  int64_t b[3];
  bool cu_in_lds, gseq_in_lds;
  const int32_t *cu, *gseq;  // cu_seqlens and the groups' first sequences there
  DEVI int64_t bound(const GaeArgs& g, int j) const {
    if (!gseq_in_lds) return group_offsets(g)[j];
    const int s = gseq[j];
    return cu_in_lds ? (int64_t)cu[s] : (int64_t)g.cu[s];
  }
};
DEVI GaeTileGroups gae_tile_groups(const GaeArgs& g, int64_t lo, const int* s_grp) {
  GaeTileGroups r;
  r.cu_in_lds = r.gseq_in_lds = false;
  r.cu = r.gseq = nullptr;
  r.g_first = s_grp[0];
  r.g_last = s_grp[1] < g.n_groups ? s_grp[1] : g.n_groups - 1;
  r.g_next = s_grp[2];
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    const int j = r.g_first + i <= g.n_groups ? r.g_first + i : g.n_groups;
    r.b[i] = group_offsets(g)[j] - lo;
  }
  return r;
}
// The same from LDS, by every wave for itself. n_lo, n_hi, n_behind: how many sequences end at or before each of the three
// tokens; a group has ended there exactly when the next one's first sequence is not among those still to come.
DEVI GaeTileGroups gae_tile_groups_lds(const GaeArgs& g, int64_t lo, bool cu_in_lds, const int32_t* cu, const int32_t* gseq,
                                       int n_lo, int n_hi, int n_behind) {
  const int lane = threadIdx.x & 63;
  GaeTileGroups r;
  r.cu_in_lds = cu_in_lds; r.gseq_in_lds = true;
  r.cu = cu; r.gseq = gseq;
  int c0 = 0, c1 = 0, c2 = 0;
  for (int j0 = 1; j0 <= g.n_groups; j0 += 64) {
    const int j = j0 + lane;
    const int s = gseq[j <= g.n_groups ? j : g.n_groups];
    c0 += __popcll(__builtin_amdgcn_ballot_w64(j <= g.n_groups && s <= n_lo));
    c1 += __popcll(__builtin_amdgcn_ballot_w64(j <= g.n_groups && s <= n_hi));
    c2 += __popcll(__builtin_amdgcn_ballot_w64(j <= g.n_groups && s <= n_behind));
  }
  r.g_first = c0;
  r.g_last = c1 < g.n_groups ? c1 : g.n_groups - 1;
  r.g_next = c2;
#pragma unroll
  for (int i = 0; i < 3; ++i) r.b[i] = r.bound(g, r.g_first + i <= g.n_groups ? r.g_first + i : g.n_groups) - lo;
  return r;
}

// Where the k-th group of the tile lies, relative to the tile's first token.
// (selects, not an index: an indexed register array would live in scratch memory)
DEVI void tile_group_bounds(const GaeArgs& g, const GaeTileGroups& tg, int64_t lo, int k, int64_t& b0, int64_t& b1) {
  auto bound = [&](int j) { return tg.bound(g, j) - lo; };
  b0 = k == 0 ? tg.b[0] : k == 1 ? tg.b[1] : k == 2 ? tg.b[2] : bound(tg.g_first + k);
  b1 = k == 0 ? tg.b[1] : k == 1 ? tg.b[2] : bound(tg.g_first + k + 1);
}
// The five masked sums of the tile's advantages per group and wave (GaeArgs::seg_stats): x = oa
// (zero for tokens outside every sequence), m = the thread's 8 mask values (zero beyond the
// array). put(group, sums) gets each wave's own, in every lane: no wave waits for another. Groups [g_begin, g_end) of
// the tile; every thread of the block calls it.
template <class Put>
DEVI void gae_tile_group_sums(const GaeArgs& g, int64_t lo, const GaeTileGroups& tg, int g_begin, int g_end,
                              const float (&oa)[GAE_ITEMS], const float (&ms)[GAE_ITEMS], const Put& put) {
  const int64_t rel = (int64_t)threadIdx.x * GAE_ITEMS;  // the thread's first token relative to lo
  // the usual 0/1 mask (decided per wave): sum m^2 = sum m, sum m^2 x = sum m x, and sum m is a count
  bool other = false;
#pragma unroll
  for (int i = 0; i < GAE_ITEMS; ++i) other |= ms[i] != 0.f && ms[i] != 1.f;
  const bool binary = __builtin_amdgcn_ballot_w64(other) == 0;
  for (int gi = g_begin; gi < g_end; ++gi) {
    // the group's bounds relative to the thread's tokens, clamped to them
    int64_t d0, d1;
    tile_group_bounds(g, tg, lo, gi - tg.g_first, d0, d1);
    d0 -= rel; d1 -= rel;
    const int i0 = d0 <= 0 ? 0 : (d0 >= GAE_ITEMS ? GAE_ITEMS : (int)d0);
    const int i1 = d1 <= 0 ? 0 : (d1 >= GAE_ITEMS ? GAE_ITEMS : (int)d1);
    double rs[5];
    if (binary) {
      int cnt = 0;
      double s1 = 0.0, s4 = 0.0;
#pragma unroll
      for (int i = 0; i < GAE_ITEMS; ++i) {
        const bool on = i >= i0 && i < i1 && ms[i] != 0.f;
        const double x = on ? (double)oa[i] : 0.0;
        cnt += on ? 1 : 0;
        s1 += x;
        s4 += x * x;
      }
      rs[0] = (double)wave_sum(cnt);
      rs[1] = wave_sum(s1);
      rs[4] = wave_sum(s4);
      rs[2] = rs[0];
      rs[3] = rs[1];
    } else {
#pragma unroll
      for (int q = 0; q < 5; ++q) rs[q] = 0.0;
#pragma unroll
      for (int i = 0; i < GAE_ITEMS; ++i) {
        const double m = (i >= i0 && i < i1) ? (double)ms[i] : 0.0;
        const double xm = (double)oa[i] * m, mm = m * m;
        rs[0] += m; rs[1] += xm; rs[2] += mm; rs[3] += xm * m; rs[4] += xm * xm;
      }
#pragma unroll
      for (int q = 0; q < 5; ++q) rs[q] = wave_sum(rs[q]);
    }
    put(gi, rs);
  }
}
DEVI void gae_tile_group_stats(const GaeArgs& g, int64_t tile, int64_t lo, int64_t hi,
                               const GaeTileGroups& tg, const float (&oa)[GAE_ITEMS],
                               const float (&ms)[GAE_ITEMS]) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int64_t st = GAE_SEG_WAVES * g.seg_slots;
  gae_tile_group_sums(g, lo, tg, tg.g_first, tg.g_last + 1, oa, ms, [&](int gi, const double (&rs)[5]) {
    if (lane == 0) {
#pragma unroll
      for (int q = 0; q < 5; ++q) g.seg_stats[(int64_t)q * st + GAE_SEG_WAVES * (tile + gi) + wave] = rs[q];
    }
  });
  // slots that no segment maps to: before the first tile's first group, between this tile's last
  // group and the next tile's first, and after the last tile's last group
  const int64_t z_lo = tile == 0 ? 0 : tile + tg.g_first;
  const int64_t r_lo = tile + tg.g_first, r_hi = tile + tg.g_last + 1;  // the slots written above
  const int64_t z_hi = hi < g.n ? tile + 1 + tg.g_next : g.seg_slots;
  for (int64_t j = GAE_SEG_WAVES * z_lo + tid; j < GAE_SEG_WAVES * z_hi; j += GAE_THREADS) {
    if (j >= GAE_SEG_WAVES * r_lo && j < GAE_SEG_WAVES * r_hi) continue;
#pragma unroll
    for (int q = 0; q < 5; ++q) g.seg_stats[(int64_t)q * st + j] = 0.0;
  }
}

// The maps of whole tiles, handed from block to block inside a launch: each wave's total, five floats and a check word made
// of them and of the call's number, each in a word of its own next to a tag made of the call's number and its place, so that a
// word says by itself whether it is this call's. A tag is half of the number, so that those of words 0, 2, 4 (1, 3, 5) of an
// earlier call fit together, by chance 2^-32: the maps of two calls often differ in b1 (word 3) alone. The check tells them all the same,
// for it starts from the half that is not in its own word's tag: of a call whose upper half fits, the lower half does not (no two
// calls have one number), and each step of the check is one to one. A wrong map takes one more chance of 2^-32, in all
// 2^-64. (Sealed as a whole like the sums, a map cost its writer and its readers a microsecond of 64-bit multiplications each.)
constexpr int GAE_LOOK_TILES = 16, MAP_WORDS = 6, MAP_PITCH = 8;  // a line of 64 bytes a wave
struct TileMaps {
  uint64_t* at;      // [tiles][GAE_SEG_WAVES][MAP_PITCH]
  uint64_t call;
  unsigned ticks;    // how long a block waits, for maps and for sums together, from when it knows its layout
  int wait;          // 0: it looks for maps once, and makes those that are not there itself
};
DEVI uint32_t map_tag(uint64_t call, int k) { return (uint32_t)(call >> (k & 1 ? 32 : 0)) + 0x9e3779b9u * (uint32_t)(k + 1); }
DEVI uint32_t map_check(uint64_t call, const MapF& m) {
  const float x[5] = {m.a11, m.a12, m.a22, m.b1, m.b2};
  uint32_t h = (uint32_t)call;
#pragma unroll
  for (int k = 0; k < 5; ++k) {
    h = (h ^ __builtin_bit_cast(uint32_t, x[k])) * 0x9e3779b1u;
    h ^= h >> 15;
  }
  return h;
}
DEVI void publish_wave_map(const TileMaps& t, int64_t tile, int wave, const MapF& m) {  // m in every lane
  const int k = threadIdx.x & 63;
  const float x = k == 0 ? m.a11 : k == 1 ? m.a12 : k == 2 ? m.a22 : k == 3 ? m.b1 : m.b2;
  const uint32_t w = k == 5 ? map_check(t.call, m) : __builtin_bit_cast(uint32_t, x);
  if (k < MAP_WORDS)
    __hip_atomic_store(t.at + (GAE_SEG_WAVES * tile + wave) * MAP_PITCH + k, (uint64_t)map_tag(t.call, k) << 32 | w,
                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// Those of n <= GAE_LOOK_TILES tiles from `first` on, by a whole wave, a lane each. False when they were not all there in time.
DEVI bool gather_tile_maps(const TileMaps& t, uint64_t deadline, int64_t first, int n, MapF* chunks) {
  const int lane = threadIdx.x & 63;
  const uint64_t* const from = t.at + (GAE_SEG_WAVES * first + lane) * MAP_PITCH;
  bool have = lane >= GAE_SEG_WAVES * n;
  for (;;) {
    if (!have) {
      uint64_t w[MAP_WORDS];
      bool all = true;
#pragma unroll
      for (int k = 0; k < MAP_WORDS; ++k) w[k] = __hip_atomic_load(from + k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
      for (int k = 0; k < MAP_WORDS; ++k) all &= (uint32_t)(w[k] >> 32) == map_tag(t.call, k);
      auto of = [&](int k) { return __builtin_bit_cast(float, (uint32_t)w[k]); };
      const MapF m{of(0), of(1), of(2), of(3), of(4)};
      if (all && (uint32_t)w[5] == map_check(t.call, m)) {
        chunks[lane] = m;
        have = true;
      }
    }
    if (__builtin_amdgcn_ballot_w64(!have) == 0) return true;
    if (wall_clock64() >= deadline) return false;
    __builtin_amdgcn_s_sleep(2);
  }
}

// STATS: tail(tile, lo, hi, groups of the tile, advantages, masks, time) gets what the group sums are made of.
// LOOK: the maps of tiles inside a crossing sequence come from their blocks, and what the tail waits for comes until `time`:
// one for both. (Read where the block starts, with no loads that it could hide behind, the clock cost 0.3 to 1.7 us.)
template <bool LAMBDAS, bool STATS, bool LOOK, class Tail>
DEVI void gae_tile(const GaeArgs& g, const TileMaps& look, const Tail& tail) {
  __shared__ MapF smem[GAE_THREADS / 64];
  __shared__ int s_grp[3];
  __shared__ MapF all[GAE_THREADS];
  __shared__ MapF s_chunk[GAE_LOOK_TILES * GAE_SEG_WAVES], s_end[GAE_SEG_WAVES];
  __shared__ int s_have;
  __shared__ int32_t s_cu[GAE_CU_LDS + 1];
  __shared__ int32_t s_gseq[STATS ? GAE_GROUPS_LDS + 1 : 1];
  __shared__ int s_own[GAE_SEG_WAVES][3];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  // XCD x (workgroup ids congruent to x modulo 8) takes the x-th eighth of the tiles
  const int64_t per_xcd = (gridDim.x + 7) >> 3;
  const int64_t tile = (int64_t)(blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
  const int64_t lo = tile * GAE_TILE;
  if (tile >= per_xcd * 8 || lo >= g.n) return;
  const int64_t hi = lo + GAE_TILE < g.n ? lo + GAE_TILE : g.n;
  // All that the block reads at its start goes out together, the layout first (loads come back in their order): the whole
  // of cu_seqlens and the groups' first sequences for LDS, and the tile's inputs.
  const bool cu_in_lds = g.n_seqs <= GAE_CU_LDS;
  const bool groups_in_lds = STATS && g.goff == nullptr && g.n_groups <= GAE_GROUPS_LDS;
  constexpr int CU_LOADS = GAE_CU_LDS / GAE_THREADS, CU_FIRST = 5, GROUP_LOADS = STATS ? GAE_GROUPS_LDS / GAE_THREADS : 1;
  int32_t c[CU_LOADS], gq[GROUP_LOADS];
  const bool many = g.n_seqs >= CU_FIRST * GAE_THREADS;  // (uniform)
  const int probe_step = (g.n_seqs + 63) >> 6;
  auto cu_of = [&](int k) { const int i = tid + k * GAE_THREADS; return g.cu[i < g.n_seqs ? i : g.n_seqs]; };  // (behind them: cov_hi)
  if (cu_in_lds) {
#pragma unroll
    for (int k = 0; k < CU_FIRST; ++k) c[k] = cu_of(k);
    if (many) {
#pragma unroll
      for (int k = CU_FIRST; k < CU_LOADS; ++k) c[k] = cu_of(k);
    }
  } else {  // the first probes of the search, which need no other load either
    c[0] = g.cu[1 + (lane * probe_step < g.n_seqs ? lane * probe_step : g.n_seqs - 1)];
  }
  if (groups_in_lds) {
#pragma unroll
    for (int k = 0; k < GROUP_LOADS; ++k) {
      const int i = tid + k * GAE_THREADS;
      if (k == 0 || k * GAE_THREADS < g.n_groups) gq[k] = (int32_t)g.gseq[i < g.n_groups ? i : g.n_groups];
    }
  }
  float rw[GAE_ITEMS], v[GAE_ITEMS], ms[GAE_ITEMS];
  gae_load_items(g, lo + (int64_t)tid * GAE_ITEMS, true, rw, v, ms);
  if constexpr (STATS) {
    if (!groups_in_lds) gae_tile_group_search(g, lo, hi, s_grp);  // (a barrier follows either way)
  }
  const int64_t cov_lo = (int64_t)g.cu[0], cov_hi = (int64_t)g.cu[g.n_seqs];
  const int64_t gseq_end = groups_in_lds ? g.gseq[g.n_groups] : 0;
  const int64_t t_begin = lo > cov_lo ? lo : cov_lo;
  const int64_t t_end = hi < cov_hi ? hi : cov_hi;
  const bool groups_from_lds = groups_in_lds && lo >= cov_lo && hi <= cov_hi;
  if constexpr (STATS) {
    if (groups_in_lds && !groups_from_lds) gae_tile_group_search(g, lo, hi, s_grp);
  }
  auto store_groups = [&] {
    if constexpr (STATS) {
      if (!groups_in_lds) return;
#pragma unroll
      for (int k = 0; k < GROUP_LOADS; ++k)
        if (k == 0 || k * GAE_THREADS < g.n_groups) s_gseq[tid + k * GAE_THREADS] = gq[k];
      if (tid == 0) s_gseq[g.n_groups] = (int32_t)gseq_end;
    }
  };
  // Sequences that end at or before the first token, the last token, and the token behind the tile.
  int n_lo = 0, n_hi = 0, n_behind = 0;
  if (cu_in_lds) {
    const int64_t top = (int64_t)INT32_MAX;
    const int32_t x0 = (int32_t)(t_begin < top ? t_begin : top), x1 = (int32_t)(t_end - 1 < top ? t_end - 1 : top),
                  x2 = (int32_t)(hi < top ? hi : top);
    auto count = [&](int k) {
      const int i = tid + k * GAE_THREADS;
      s_cu[i] = c[k];
      const bool end = i >= 1 && i < g.n_seqs;
      n_lo += __popcll(__builtin_amdgcn_ballot_w64(end && c[k] <= x0));
      n_hi += __popcll(__builtin_amdgcn_ballot_w64(end && c[k] <= x1));
      if constexpr (STATS) n_behind += __popcll(__builtin_amdgcn_ballot_w64(end && c[k] <= x2));
    };
#pragma unroll
    for (int k = 0; k < CU_FIRST; ++k) count(k);
    if (many) {
#pragma unroll
      for (int k = CU_FIRST; k < CU_LOADS; ++k) count(k);
    }
    store_groups();
    if (tid == 0) {  // the last entry
      s_cu[g.n_seqs] = (int32_t)cov_hi;
      n_lo += (int32_t)cov_hi <= x0;
      n_hi += (int32_t)cov_hi <= x1;
      if constexpr (STATS) n_behind += (int32_t)cov_hi <= x2;
    }
    if (lane == 0) { s_own[wave][0] = n_lo; s_own[wave][1] = n_hi; s_own[wave][2] = n_behind; }
    __syncthreads();
    n_lo = n_hi = n_behind = 0;
#pragma unroll
    for (int w = 0; w < GAE_SEG_WAVES; ++w) { n_lo += s_own[w][0]; n_hi += s_own[w][1]; n_behind += s_own[w][2]; }
  }
  // tokens outside every sequence (none in a well-formed batch) are written as zero
  if (lo < cov_lo || hi > cov_hi) {
    for (int64_t t = lo + tid; t < hi; t += GAE_THREADS)
      if (t < cov_lo || t >= cov_hi) { g.adv[t] = 0.f; g.ret[t] = 0.f; }
  }
  const bool none = t_end <= t_begin;  // no token of a sequence (uniform for the block)
  if (!STATS && none) return;

  // sequences holding the first and the last token of [t_begin, t_end)
  const int32_t* cu_own;
  int s_first, s_last;
  if (cu_in_lds) {
    s_first = __builtin_amdgcn_readfirstlane(n_lo);
    s_last = __builtin_amdgcn_readfirstlane(n_hi);
    cu_own = s_cu + s_first;
  } else {
    if (wave == GAE_SEG_WAVES - 1) {  // (the one that searches for no group, where groups are searched for)
      const int hits = __popcll(__builtin_amdgcn_ballot_w64(lane * probe_step < g.n_seqs && (int64_t)c[0] <= t_begin));
      const int most = hits > 0 ? probe_step - 1 : 0;
      int from = hits > 0 ? (hits - 1) * probe_step + 1 : 0;
      if (probe_step > 64) from += wave_count_le(g.cu + 1 + from, most < g.n_seqs - from ? most : g.n_seqs - from, t_begin, lane);
      // cu_seqlens from `from` on: the first token's sequence is one of the next 64, and as a rule all that the tile has to
      // know follows within 64 more
      const int i0 = from + lane, i1 = i0 + 64;
      const int32_t e0 = g.cu[i0 < g.n_seqs ? i0 : g.n_seqs], e1 = g.cu[i1 < g.n_seqs ? i1 : g.n_seqs];
      auto ended = [&](int64_t x) {
        return from + __popcll(__builtin_amdgcn_ballot_w64(lane > 0 && i0 <= g.n_seqs && (int64_t)e0 <= x)) +
               __popcll(__builtin_amdgcn_ballot_w64(i1 <= g.n_seqs && (int64_t)e1 <= x));
      };
      const int r = ended(t_begin);
      int l = ended(t_end - 1), b = STATS ? ended(hi) : 0;
      const bool held = l < from + 127;
      if (!held) l += wave_count_le(g.cu + 1 + l, g.n_seqs - l, t_end - 1, lane);
      if (STATS && b == from + 127) b += wave_count_le(g.cu + 1 + b, g.n_seqs - b, hi, lane);
      if (held) {
        if (i0 >= r && i0 <= l + 1) s_cu[i0 - r] = e0;
        if (i1 >= r && i1 <= l + 1) s_cu[i1 - r] = e1;
      }
      if (lane == 0) { s_own[0][0] = r; s_own[0][1] = l; s_own[0][2] = b; s_own[1][0] = held; }
    }
    store_groups();
    __syncthreads();
    s_first = __builtin_amdgcn_readfirstlane(s_own[0][0]);
    s_last = __builtin_amdgcn_readfirstlane(s_own[0][1]);
    n_behind = s_own[0][2];
    if (none) {
      cu_own = g.cu;  // (not read: behind the last sequence there is no next entry)
    } else if (s_own[1][0] != 0) {
      cu_own = s_cu;
    } else if (s_last - s_first + 1 <= GAE_CU_LDS) {
      for (int i = tid; i <= s_last - s_first + 1; i += GAE_THREADS) s_cu[i] = g.cu[s_first + i];
      __syncthreads();
      cu_own = s_cu;
    } else {
      cu_own = g.cu + s_first;  // only with many empty sequences
    }
  }
  const int n_own = s_last - s_first + 1;
  GaeTileGroups tg;
  if constexpr (STATS) {
    tg = groups_from_lds ? gae_tile_groups_lds(g, lo, cu_in_lds, s_cu, s_gseq, s_first, s_last, n_behind)
                         : gae_tile_groups(g, lo, s_grp);
  }
  const uint64_t deadline = LOOK ? wall_clock64() + look.ticks : 0;

  // The crossing sequence's tokens [t_end, e) lie in `full` whole tiles and the tile with its last token. Their maps, a wave's
  // chunk of 512 tokens at a time, are applied in fp64 one after the other from the right: those of the last tile made here,
  // those of whole tiles taken from the blocks of these tiles (LOOK), or made here as well; the same numbers either way.
  double A0 = 0.0, nv0 = 0.0;
  const int64_t e = none ? 0 : (int64_t)cu_own[n_own];
  if (e > t_end) {
    const int64_t last_tile = (e - 1) / GAE_TILE;
    const int full = (int)(last_tile - tile) - 1;
    const float gam = g.discount;
    const float c = gam * (LAMBDAS ? g.lam_seq[s_last] : g.lam);
    const bool boot = g.no_eos != nullptr && g.no_eos[s_last] != 0;
    // (without values the mask is read in their place and dropped: no branch between the loads)
    const float* const values = g.values != nullptr ? g.values : g.mask;
    auto token_of = [&](int64_t from, int k) { return from * GAE_TILE + k * GAE_CHUNK + (int64_t)lane * GAE_ITEMS; };
    float crw[GAE_ITEMS], cv[GAE_ITEMS], cms[GAE_ITEMS];
    auto fetch = [&](int64_t t0) {
      if (t0 + GAE_ITEMS <= g.n) {
#pragma unroll
        for (int q = 0; q < GAE_ITEMS / 4; ++q) {
          const f32x4 a = *(const f32x4*)(g.rewards + t0 + 4 * q);
          const f32x4 b = *(const f32x4*)(values + t0 + 4 * q);
          const f32x4 m = *(const f32x4*)(g.mask + t0 + 4 * q);
#pragma unroll
          for (int x = 0; x < 4; ++x) { crw[4 * q + x] = a[x]; cv[4 * q + x] = b[x]; cms[4 * q + x] = m[x]; }
        }
      } else {
#pragma unroll
        for (int i = 0; i < GAE_ITEMS; ++i) {
          const bool in = t0 + i < g.n;
          crw[i] = in ? g.rewards[t0 + i] : 0.f;
          cv[i] = in ? values[t0 + i] : 0.f;
          cms[i] = in ? g.mask[t0 + i] : 0.f;
        }
      }
      if (g.values == nullptr) {
#pragma unroll
        for (int i = 0; i < GAE_ITEMS; ++i) cv[i] = 0.f;
      }
    };
    // whole: of a tile inside the sequence (its last token lies in a later one)
    auto chunk_map = [&](auto whole, int64_t t0, const float (&r)[GAE_ITEMS], const float (&val)[GAE_ITEMS],
                         const float (&mask)[GAE_ITEMS]) {
      constexpr bool WHOLE = decltype(whole)::value;
      const int left = e - t0 < 2 * GAE_ITEMS ? (int)(e - t0) : 2 * GAE_ITEMS;  // the thread's tokens of the sequence
      MapF acc = map_identity_t<float>();
#pragma unroll
      for (int i = GAE_ITEMS - 1; i >= 0; --i) {
        // beyond the sequence (or the batch): identity; its last token: the constant map
        const float m = WHOLE || i < left ? mask[i] : 0.f;
        MapF f;
        f.a11 = fmaf(c, m, 1.f - m);
        f.a12 = gam * m;
        f.a22 = 1.f - m;
        f.b1 = (r[i] - val[i]) * m;
        f.b2 = val[i] * m;
        if (!WHOLE && i == left - 1) f = MapF{0.f, 0.f, 0.f, 0.f, boot ? val[i] : 0.f};
        acc = compose(f, acc);
      }
      return wave_total_map(acc);
    };
    auto apply = [&](const MapF& m) {
      const double A1 = fma((double)m.a11, A0, fma((double)m.a12, nv0, (double)m.b1));
      nv0 = fma((double)m.a22, nv0, (double)m.b2);
      A0 = A1;
    };
    float xr[GAE_ITEMS], xv[GAE_ITEMS], xm[GAE_ITEMS];
    auto take = [&] {
#pragma unroll
      for (int i = 0; i < GAE_ITEMS; ++i) { xr[i] = crw[i]; xv[i] = cv[i]; xm[i] = cms[i]; }
    };
    // whole tiles from the right, GAE_LOOK_TILES at a time
    bool ask = LOOK;  // until one wait was in vain
    int right = full, n = right < GAE_LOOK_TILES ? right : GAE_LOOK_TILES;
    int64_t first = tile + 1 + right - n;
    const bool in_end = last_tile * GAE_TILE + wave * GAE_CHUNK < e;  // the wave's chunk of the last tile holds tokens of it
    if (in_end) fetch(token_of(last_tile, wave));
    if constexpr (LOOK) {
      // a tile inside one sequence that goes on behind it: tiles on its left may want its maps
      if (n_own == 1 && (int64_t)cu_own[0] < lo)
        publish_wave_map(look, tile, wave, chunk_map(std::true_type{}, lo + (int64_t)tid * GAE_ITEMS, rw, v, ms));
    }
    take();
    if (!ask && n > 0) fetch(token_of(first, wave));  // on its way meanwhile
    {
      MapF m = map_identity_t<float>();
      if (in_end) m = chunk_map(std::false_type{}, token_of(last_tile, wave), xr, xv, xm);
      if (lane == 0) s_end[wave] = m;
    }
    for (bool at_end = true;; at_end = false) {  // uniform for the block
      bool have = n == 0;
      if (ask) {
        if (!have && wave == 0) {
          const bool all_there = gather_tile_maps(look, look.wait ? deadline : 0, first, n, s_chunk);
          if (lane == 0) s_have = all_there ? 1 : 0;
        }
        __syncthreads();
        have = have || s_have != 0;
        if (!have) { ask = false; fetch(token_of(first, wave)); }
      }
      if (!have) {
        for (int k = wave; k < n * GAE_SEG_WAVES; k += GAE_SEG_WAVES) {
          take();
          if (k + GAE_SEG_WAVES < n * GAE_SEG_WAVES) fetch(token_of(first, k + GAE_SEG_WAVES));
          const MapF m = chunk_map(std::true_type{}, token_of(first, k), xr, xv, xm);
          if (lane == 0) s_chunk[k] = m;
        }
      }
      if (!ask) __syncthreads();
      if (at_end) {
#pragma unroll
        for (int w = GAE_SEG_WAVES - 1; w >= 0; --w) apply(s_end[w]);
      }
      for (int t = n - 1; t >= 0; --t) {
        MapF m[GAE_SEG_WAVES];  // (read together: the chain is that of the products alone)
#pragma unroll
        for (int w = 0; w < GAE_SEG_WAVES; ++w) m[w] = s_chunk[t * GAE_SEG_WAVES + w];
#pragma unroll
        for (int w = GAE_SEG_WAVES - 1; w >= 0; --w) apply(m[w]);
      }
      right -= n;
      if (right <= 0) break;
      n = right < GAE_LOOK_TILES ? right : GAE_LOOK_TILES;
      first = tile + 1 + right - n;
      if (!ask) fetch(token_of(first, wave));
      __syncthreads();  // s_chunk has been read
    }
  }
  float oa[GAE_ITEMS];
  if (none) {
#pragma unroll
    for (int i = 0; i < GAE_ITEMS; ++i) oa[i] = 0.f;
  } else {
    gae_one_tile<GAE_LAYOUT_CU, LAMBDAS>(g, tile, t_begin, t_end, s_first, n_own, cu_own, A0, nv0, smem, all, rw, v, ms, oa);
  }
  if constexpr (STATS) tail(tile, lo, hi, tg, oa, ms, deadline);
}
// STATS: also leaves the per-(tile, group) sums of GaeArgs::seg_stats.
template <bool LAMBDAS, bool STATS>
__global__ __launch_bounds__(GAE_THREADS, 4) void gae_tile_kernel(GaeArgs g) {
  gae_tile<LAMBDAS, STATS, false>(g, TileMaps{}, [&](int64_t tile, int64_t lo, int64_t hi, const GaeTileGroups& tg, const float (&oa)[GAE_ITEMS],
                                  const float (&ms)[GAE_ITEMS], uint64_t) { gae_tile_group_stats(g, tile, lo, hi, tg, oa, ms); });
}

// ---------------------------------------------------------------------------------------
// Normalisation
// ---------------------------------------------------------------------------------------
constexpr int NORM_THREADS = 256;
constexpr int SEG_APPLY_ELEMS = 16 * NORM_THREADS;  // elements per block of the apply pass after the packed GAE
enum { LEVEL_NONE = 0, LEVEL_BATCH = 1, LEVEL_GROUP = 2 };

struct NormArgs {
  const float* x;
  const float* mask;       // nullable
  int64_t n;
  const int64_t* goff;     // [G+1] element offsets of the groups (cover [0, n))
  const int64_t* grows;    // [G] rows in each group (for the singleton rules)
  int G;
  int tail_group;          // index of the group holding ungrouped tail rows, or -1
  int nsplit;              // blocks per group
  int mean_level, std_level;
  int leave1out, unbiased;
  double eps;
  double* part;            // [3][G][nsplit]: count, sum, sum of squared deviations; or, with
                           // closed_form, [5][G][nsplit]: sum m, sum x m, sum m^2, sum m^2 x, sum m^2 x^2
  float* out;
  int closed_form;         // the squared deviations come from the five sums of one statistics pass
  // closed form only: where the five sums of a group are. part_rows == 0: [5][G][nsplit], written
  // by norm_stats5_kernel. part_rows > 0: [5][part_rows], one entry per row of row_len elements
  // (written by the GAE kernel); group g owns the rows from goff[g] / row_len on, grows[g] of them.
  // part_tile > 0: [5][part_slots][4], four entries per (tile of part_tile tokens, group) segment
  // in slot tile + group (written by the packed GAE kernel, GaeArgs::seg_stats); unused slots are zero.
  int64_t part_rows, row_len;
  int64_t part_tile, part_slots;
};

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

DEVI void split_range(const NormArgs& a, int g, int sp, int64_t& lo, int64_t& hi) {
  const int64_t g0 = a.goff[g], g1 = a.goff[g + 1];
  const int64_t len = g1 - g0;
  const int64_t per = (len + a.nsplit - 1) / a.nsplit;
  lo = g0 + (int64_t)sp * per;
  hi = lo + per;
  if (hi > g1) hi = g1;
  if (lo > g1) lo = g1;
}

// Sum of one partial array over all splits of group g, computed cooperatively by the block
// (fixed order: the same tree whatever the launch).
DEVI double group_partial(const NormArgs& a, int which, int g, double* smem) {
  double r = 0.0;
  const double* p = a.part + ((int64_t)which * a.G + g) * a.nsplit;
  for (int i = threadIdx.x; i < a.nsplit; i += blockDim.x) r += p[i];
  return block_sum_d(r, smem);
}
// Sum over every group and split, computed cooperatively by the block.
DEVI double batch_partial(const NormArgs& a, int which, double* smem) {
  double r = 0.0;
  const double* p = a.part + (int64_t)which * a.G * a.nsplit;
  const int64_t tot = (int64_t)a.G * a.nsplit;
  for (int64_t i = threadIdx.x; i < tot; i += blockDim.x) r += p[i];
  return block_sum_d(r, smem);
}

struct MeanCtx {
  int level;      // LEVEL_*
  bool identity;  // singleton group with leave-one-out: mean = x
  bool zero;      // tail group, or leave-one-out with count <= 1, or empty: mean = 0
  bool loo;
  double cnt, sum;
};

DEVI MeanCtx make_mean_ctx(const NormArgs& a, int g, double* smem) {
  MeanCtx c;
  c.level = a.mean_level; c.identity = false; c.zero = false; c.loo = a.leave1out != 0;
  c.cnt = 0.0; c.sum = 0.0;
  if (a.mean_level == LEVEL_BATCH) {
    c.cnt = batch_partial(a, 0, smem);
    c.sum = batch_partial(a, 1, smem);
  } else if (a.mean_level == LEVEL_GROUP) {
    if (g == a.tail_group) { c.zero = true; return c; }
    if (a.grows[g] == 1 && c.loo) { c.identity = true; return c; }
    c.cnt = group_partial(a, 0, g, smem);
    c.sum = group_partial(a, 1, g, smem);
  } else {
    c.zero = true;
    return c;
  }
  if (c.loo) { if (c.cnt <= 1.0) c.zero = true; }
  else if (c.cnt == 0.0) c.zero = true;
  return c;
}

// Mean seen by one element, as the reference stores it: group-level means are rounded to
// fp32 (they are written into a zeros_like(x) tensor), batch-level means stay fp64.
DEVI double elem_mean(const MeanCtx& c, float x, float m, bool has_mask) {
  double mean;
  if (c.zero) mean = 0.0;
  else if (c.identity) mean = (double)x;
  else if (!c.loo) mean = c.sum / c.cnt;
  else if (!has_mask) mean = (c.sum - (double)x) / (c.cnt - 1.0);
  else {
    const double md = (double)m;
    if (md > 0.0) {
      double den = c.cnt - md;
      if (den < 1.0) den = 1.0;
      mean = (c.sum - (double)x * md) / den;
    } else {
      mean = c.sum / c.cnt;
    }
  }
  if (c.level != LEVEL_BATCH) mean = (double)(float)mean;
  return mean;
}

// pass 1: count and sum per (group, split)
__global__ __launch_bounds__(NORM_THREADS) void norm_stats1_kernel(NormArgs a) {
  __shared__ double smem[4];
  const int g = blockIdx.x, sp = blockIdx.y;
  int64_t lo, hi;
  split_range(a, g, sp, lo, hi);
  double cnt = 0.0, sum = 0.0;
  for (int64_t i = lo + threadIdx.x; i < hi; i += blockDim.x) {
    const double m = a.mask ? (double)a.mask[i] : 1.0;
    cnt += m;
    sum += (double)a.x[i] * m;
  }
  cnt = block_sum_d(cnt, smem);
  sum = block_sum_d(sum, smem);
  if (threadIdx.x == 0) {
    a.part[((int64_t)0 * a.G + g) * a.nsplit + sp] = cnt;
    a.part[((int64_t)1 * a.G + g) * a.nsplit + sp] = sum;
  }
}

// The only statistics pass of the two-launch form: five masked sums per (group, split). With a
// mean that is the same for every element of a group (no leave-one-out), the sum of squared
// deviations sum (x m - mean m)^2 is S(m^2 x^2) - 2 mean S(m^2 x) + mean^2 S(m^2), evaluated in
// fp64 by the apply pass with the mean exactly as the elements see it (rounded to fp32 at group
// level), so x and the mask are read once for the statistics instead of twice.
__global__ __launch_bounds__(NORM_THREADS) void norm_stats5_kernel(NormArgs a) {
  __shared__ double smem[4 * 5];
  const int g = blockIdx.x, sp = blockIdx.y;
  int64_t lo, hi;
  split_range(a, g, sp, lo, hi);
  double s0 = 0.0, s1 = 0.0, s2 = 0.0, s3 = 0.0, s4 = 0.0;
  auto take = [&](float xf, float mf) {
    const double x = (double)xf, m = (double)mf;
    const double xm = x * m, mm = m * m;
    s0 += m; s1 += xm; s2 += mm; s3 += xm * m; s4 += xm * xm;
  };
  const bool has_mask = a.mask != nullptr;
  // scalar head up to a multiple of 4 elements, 16-byte loads in the middle, scalar tail
  int64_t mid_lo = (lo + 3) & ~(int64_t)3, mid_hi = hi & ~(int64_t)3;
  if (mid_lo > mid_hi) { mid_lo = hi; mid_hi = hi; }
  for (int64_t i = lo + threadIdx.x; i < mid_lo; i += blockDim.x) take(a.x[i], has_mask ? a.mask[i] : 1.0f);
  // four 16-byte loads of each array in flight per thread before the first sum needs them
  const int64_t step = 4 * (int64_t)blockDim.x;
  for (int64_t i = mid_lo + 4 * (int64_t)threadIdx.x; i < mid_hi; i += 4 * step) {
    f32x4 xv[4], mv[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int64_t j = i + u * step;
      xv[u] = f32x4{0.f, 0.f, 0.f, 0.f};
      mv[u] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (j < mid_hi) {
        xv[u] = *(const f32x4*)(a.x + j);
        mv[u] = has_mask ? *(const f32x4*)(a.mask + j) : f32x4{1.f, 1.f, 1.f, 1.f};
      }
    }
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int e = 0; e < 4; ++e) take(xv[u][e], mv[u][e]);
  }
  for (int64_t i = mid_hi + threadIdx.x; i < hi; i += blockDim.x)
    if (i >= mid_lo) take(a.x[i], has_mask ? a.mask[i] : 1.0f);
  double v[5] = {s0, s1, s2, s3, s4};
  block_sum_n<5>(v, smem);
  if (threadIdx.x == 0) {
    const int64_t o = (int64_t)g * a.nsplit + sp, st = (int64_t)a.G * a.nsplit;
#pragma unroll
    for (int k = 0; k < 5; ++k) a.part[k * st + o] = v[k];
  }
}

// What the elements of group g are normalised with, from the five sums of the group (v[0..4]) and of the
// batch (v[5..9]; only v[5] unless a level is "batch"); no leave-one-out here.
struct NormParams {
  double mean, std_d, eps;
  bool mean64, std64;
};
// rows(): the number of rows of the group (asked for only where it counts).
template <class Rows>
DEVI NormParams norm_params(const NormArgs& a, int g, const double (&v)[10], const Rows& rows) {
  // mean context (see make_mean_ctx)
  MeanCtx mc;
  mc.level = a.mean_level; mc.identity = false; mc.zero = false; mc.loo = false; mc.cnt = 0.0; mc.sum = 0.0;
  if (a.mean_level == LEVEL_BATCH) { mc.cnt = v[5]; mc.sum = v[6]; if (mc.cnt == 0.0) mc.zero = true; }
  else if (a.mean_level == LEVEL_GROUP) {
    if (g == a.tail_group) mc.zero = true;
    else { mc.cnt = v[0]; mc.sum = v[1]; if (mc.cnt == 0.0) mc.zero = true; }
  } else mc.zero = true;
  NormParams np;
  np.mean = elem_mean(mc, 0.f, 1.f, false);  // one value for the whole group
  const double mean = np.mean;
  auto ss_of = [&](double s2, double s3, double s4) {
    const double ss = s4 - 2.0 * mean * s3 + mean * mean * s2;
    return ss > 0.0 ? ss : 0.0;
  };
  double std_d = 1.0;
  np.eps = a.eps;
  if (a.std_level == LEVEL_BATCH) {
    const double cnt = v[5], ss = ss_of(v[7], v[8], v[9]);
    if (a.unbiased) std_d = cnt <= 1.0 ? 1.0 : sqrt(ss / (cnt - 1.0));
    else std_d = cnt == 0.0 ? 1.0 : sqrt(ss / cnt);
  } else if (a.std_level == LEVEL_GROUP) {
    if (g == a.tail_group) std_d = 0.0;
    else if (a.unbiased && rows() == 1) std_d = 1.0;
    else {
      const double cnt = v[0], ss = ss_of(v[2], v[3], v[4]);
      if (a.unbiased) std_d = cnt <= 1.0 ? 1.0 : sqrt(ss / (cnt - 1.0));
      else std_d = cnt == 0.0 ? 1.0 : sqrt(ss / cnt);
    }
    std_d = (double)(float)std_d;
  } else {
    np.eps = 0.0;
  }
  np.std_d = std_d;
  np.mean64 = a.mean_level == LEVEL_BATCH;
  np.std64 = a.std_level == LEVEL_BATCH;
  return np;
}
DEVI NormParams norm_params(const NormArgs& a, int g, const double (&v)[10]) {
  return norm_params(a, g, v, [&] { return a.grows[g]; });
}
DEVI float norm_one(const NormParams& p, float x, float m, bool has_mask) {
  if (p.mean64 || p.std64) {
    double c = p.mean64 ? ((double)x - p.mean) : (double)(x - (float)p.mean);
    if (has_mask) c = p.mean64 ? c * (double)m : (double)((float)c * m);
    const double den = p.std64 ? (p.std_d + p.eps) : (double)((float)p.std_d + (float)p.eps);
    return (float)(c / den);
  }
  float c = x - (float)p.mean;
  if (has_mask) c = c * m;
  return c / ((float)p.std_d + (float)p.eps);
}

// ---- Packed GAE and the normalisation of its advantages within groups of sequences in one launch: a tile's block keeps its
// advantages in registers, publishes its sums per group and waits for those of the other tiles of its groups, each
// wave for another group. A launch of its own read advantages and masks back and searched the groups again, several loads
// that wait for each other. Two launches / one, GAE included, us: 1024 sequences of 1750 tokens in groups of 16 28.1 / 25.1, 4096 of
// 100 in fours (five groups to a tile) 56.0 / 34.0, 64 of 300 17.1 / 14.5, 64 of 8192 in eights 40.1 / 18.8 (equal lengths 16.8 /
// 15.3). The rule for the sizes of groups stands at areal_gae_packed_normalized_ex.
// No wait is unbounded, as with adv_normalise_row, and maps and sums have one time together: when it is up, the block leaves a note for the (tile, group)
// segment, whose advantages are in memory anyway, and a wave that finds all sums of a group looks for notes of its tiles and
// takes them. Leaving a note is followed by another look at the sums, publishing comes before the look for notes (leave_note).
// Where not all tiles are on the chip at once, only the last GAE_WAIT_TILES tiles of a group on an XCD wait (it holds 128), the
// ones before them leave a note at once: all of them waiting would keep the last ones from starting until the time is up, and
// those would find every note alone. The rule at areal_gae_packed_normalized_ex goes by average lengths, and one group may be far
// longer. 3200 sequences of 700 tokens and a group of 195 tiles, us: behind them 441 -> 172, in front 491 -> 195, in the middle
// 112 (two launches 118, 133, 119); a group of 78 tiles 52 (64), eight of 117 126 (109).
constexpr int GAE_TILES_AT_ONCE = 1024, GAE_WAIT_TILES = 112;
constexpr int SUMS_PITCH = 8;  // words an entry: five sums, their seal, a line of 64 bytes to itself
struct GaeNormArgs {
  GaeArgs g;
  NormArgs norm;              // levels; out: the normalised advantages
  uint64_t *sums, *flags, *left;  // [seg_slots][SUMS_PITCH] and twice [seg_slots] in the workspace
  uint64_t call;
  TileMaps maps;
};
DEVI void gae_tile_normalise(const GaeNormArgs& a, uint64_t deadline, int64_t tile, int64_t lo, int64_t hi, const GaeTileGroups& tg,
                             const float (&oa)[GAE_ITEMS], const float (&ms)[GAE_ITEMS]) {
  __shared__ double s_sum[GAE_SEG_WAVES][GAE_SEG_WAVES][5];  // [group][wave]
  __shared__ float s_mean[GAE_SEG_WAVES], s_den[GAE_SEG_WAVES];
  __shared__ int s_lo[GAE_SEG_WAVES], s_hi[GAE_SEG_WAVES], s_state[GAE_SEG_WAVES];
  constexpr int NONE = 0, READY = 1, LEFT = 2;
  const GaeArgs& g = a.g;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, rel = tid * GAE_ITEMS;
  auto entry = [&](int64_t k, int gi) { return a.sums + SUMS_PITCH * (k + gi); };
  for (int gb = tg.g_first; gb <= tg.g_last; gb += GAE_SEG_WAVES) {
    const int g_end = gb + GAE_SEG_WAVES <= tg.g_last + 1 ? gb + GAE_SEG_WAVES : tg.g_last + 1;
    gae_tile_group_sums(g, lo, tg, gb, g_end, oa, ms, [&](int gi, const double (&rs)[5]) {
      if (lane == 0) {
#pragma unroll
        for (int k = 0; k < 5; ++k) s_sum[gi - gb][wave][k] = rs[k];
      }
    });
    __syncthreads();
    if (lane == 0 && gb + wave < g_end) {
      double rs[5];
#pragma unroll
      for (int k = 0; k < 5; ++k)
        rs[k] = (s_sum[wave][0][k] + s_sum[wave][1][k]) + (s_sum[wave][2][k] + s_sum[wave][3][k]);
      publish_sums(entry(tile, gb + wave), a.flags + tile + gb + wave, a.call, rs);
    }
    if (gb + GAE_SEG_WAVES <= tg.g_last) __syncthreads();
  }
  const int64_t per_xcd = (gridDim.x + 7) >> 3, xcd_last = ((blockIdx.x & 7) + 1) * per_xcd - 1;
  float r[GAE_ITEMS];
  unsigned keep = 0;  // tokens of groups that were left
#pragma unroll
  for (int i = 0; i < GAE_ITEMS; ++i) r[i] = 0.f;  // (a token of no group is one of no sequence)
  for (int gb = tg.g_first; gb <= tg.g_last; gb += GAE_SEG_WAVES) {
    const int gi = gb + wave;
    int64_t b0 = 0, b1 = 0;  // the wave's group, relative to the tile
    if (gi <= tg.g_last) tile_group_bounds(g, tg, lo, gi - tg.g_first, b0, b1);
    const bool mine = b0 < b1;
    const int64_t rows = mine ? a.norm.grows[gi] : 0;
    const int64_t k0 = (lo + b0) / GAE_TILE, k1 = (lo + b1 - 1) / GAE_TILE;
    float mean = 0.f, den = 1.f;
    auto gather = [&](uint64_t until) {
      double s[5], v[10];
      if (!gather_sums<SUMS_PITCH>(entry(k0, gi), a.flags + k0 + gi, (int)(k1 - k0 + 1), a.call, until, s)) return false;
#pragma unroll
      for (int k = 0; k < 5; ++k) { v[k] = s[k]; v[5 + k] = 0.0; }
      const NormParams np = norm_params(a.norm, gi, v, [&] { return rows; });
      mean = (float)np.mean;
      den = (float)np.std_d + (float)np.eps;
      return true;
    };
    auto take_notes = [&] {  // of the wave's group
      published_before_notes();
      for (int64_t kb = k0; kb <= k1; kb += 64) {
        for (;;) {
          const uint64_t notes = __builtin_amdgcn_ballot_w64(kb + lane <= k1 && note_left(a.left + kb + lane + gi, a.call));
          if (notes == 0) break;
          // (from the wave's own place on: of those that look together not all try for the same one)
          const uint64_t behind = notes & (~0ull << (tile & 63));
          const int64_t k = kb + __builtin_ctzll(behind != 0 ? behind : notes);
          int got = 0;
          if (lane == 0) got = take_note(a.left + k + gi, a.call) ? 1 : 0;
          if (__builtin_amdgcn_readfirstlane(got) == 0) continue;  // somebody else's
          __threadfence();
          const int64_t s0 = k * GAE_TILE > lo + b0 ? k * GAE_TILE : lo + b0;
          const int64_t s1 = (k + 1) * GAE_TILE < lo + b1 ? (k + 1) * GAE_TILE : lo + b1;
          for (int64_t t = s0 + lane; t < s1; t += 64) {
            const float c = (g.adv[t] - mean) * g.mask[t];
            a.norm.out[t] = c / den;
          }
        }
      }
    };
    const int64_t to_come = (k1 < xcd_last ? k1 : xcd_last) - tile;  // on this XCD
    const bool patient = gridDim.x <= GAE_TILES_AT_ONCE || to_come < GAE_WAIT_TILES;
    const bool ready = mine && gather(patient ? deadline : 0);
    if (lane == 0) {
      s_mean[wave] = mean;
      s_den[wave] = den;
      s_lo[wave] = (int)(b0 > 0 ? b0 : 0);
      s_hi[wave] = (int)(b1 < GAE_TILE ? b1 : GAE_TILE);
      s_state[wave] = !mine ? NONE : ready ? READY : LEFT;
    }
    __syncthreads();
    bool left = false;
    for (int w = 0; w < GAE_SEG_WAVES; ++w) {
      if (s_state[w] == NONE) continue;
      const float wm = s_mean[w], wd = s_den[w];
      const int i0 = s_lo[w] - rel, i1 = s_hi[w] - rel;
      left |= s_state[w] == LEFT;
#pragma unroll
      for (int i = 0; i < GAE_ITEMS; ++i) {
        if (i < i0 || i >= i1) continue;
        if (s_state[w] == LEFT) keep |= 1u << i;
        else r[i] = (oa[i] - wm) * ms[i] / wd;
      }
    }
    __syncthreads();
    if (ready) take_notes();
    if (left) {
      __threadfence();  // the block's advantages are in memory
      __syncthreads();
      if (mine && !ready) {
        if (lane == 0) leave_note(a.left + tile + gi, a.call);
        if (gather(0)) take_notes();
      }
    }
  }
  const int64_t t0 = lo + rel;
  if (keep == 0 && t0 + GAE_ITEMS <= hi) {
#pragma unroll
    for (int q = 0; q < GAE_ITEMS / 4; ++q)
      *(f32x4_any*)(a.norm.out + t0 + 4 * q) = f32x4{r[4 * q], r[4 * q + 1], r[4 * q + 2], r[4 * q + 3]};
  } else {
#pragma unroll
    for (int i = 0; i < GAE_ITEMS; ++i)
      if (t0 + i < hi && ((keep >> i) & 1u) == 0) a.norm.out[t0 + i] = r[i];
  }
}
template <bool LAMBDAS>
__global__ __launch_bounds__(GAE_THREADS, 4) void gae_tile_norm_kernel(GaeNormArgs a) {
  gae_tile<LAMBDAS, true, true>(a.g, a.maps, [&](int64_t tile, int64_t lo, int64_t hi, const GaeTileGroups& tg, const float (&oa)[GAE_ITEMS],
                                   const float (&ms)[GAE_ITEMS], uint64_t deadline) { gae_tile_normalise(a, deadline, tile, lo, hi, tg, oa, ms); });
}

// Apply pass of the two-launch form. Every block first sums what it needs of the five partial
// arrays in one cooperative sweep (its group's five sums; the batch's count, or all five batch
// sums when a level is "batch") and one fused block reduction, then derives the mean and the
// deviation exactly as the three-launch kernels do, and streams its range with 16-byte accesses.
__global__ __launch_bounds__(NORM_THREADS) void norm_apply_cf_kernel(NormArgs a) {
  __shared__ double smem[4 * 10];
  const int g = blockIdx.x, sp = blockIdx.y;
  const bool has_mask = a.mask != nullptr;
  int64_t lo, hi;
  split_range(a, g, sp, lo, hi);
  const bool any_batch = a.mean_level == LEVEL_BATCH || a.std_level == LEVEL_BATCH;
  // The block's first 16 elements per thread are requested before the partial sums, which then
  // arrive while those loads are in flight.
  int64_t mid_lo = (lo + 3) & ~(int64_t)3, mid_hi = hi & ~(int64_t)3;
  if (mid_lo > mid_hi) { mid_lo = hi; mid_hi = hi; }
  const int64_t step = 4 * (int64_t)blockDim.x;
  f32x4 xv[4], mv[4];
  auto fetch = [&](int64_t i) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int64_t j = i + u * step;
      xv[u] = f32x4{0.f, 0.f, 0.f, 0.f};
      mv[u] = f32x4{1.f, 1.f, 1.f, 1.f};
      if (j < mid_hi) {
        xv[u] = *(const f32x4*)(a.x + j);
        if (has_mask) mv[u] = *(const f32x4*)(a.mask + j);
      }
    }
  };
  const int64_t i0 = mid_lo + 4 * (int64_t)threadIdx.x;
  fetch(i0);
  int64_t st, p0, pn;  // the group's partial sums: entries [p0, p0 + pn) of arrays of st entries
  if (a.part_tile > 0) {
    const int64_t g0 = a.goff[g], g1 = a.goff[g + 1];
    st = GAE_SEG_WAVES * a.part_slots;
    p0 = GAE_SEG_WAVES * (g0 / a.part_tile + g);
    pn = g1 > g0 ? GAE_SEG_WAVES * ((g1 - 1) / a.part_tile - g0 / a.part_tile + 1) : 0;
  } else if (a.part_rows > 0) {
    st = a.part_rows;
    p0 = a.goff[g] / a.row_len;
    pn = g == a.tail_group ? a.part_rows - p0 : a.grows[g];
  } else {
    st = (int64_t)a.G * a.nsplit;
    p0 = (int64_t)g * a.nsplit;
    pn = a.nsplit;
  }
  double v[10];  // group sums 0..4, batch sums 5..9
#pragma unroll
  for (int k = 0; k < 10; ++k) v[k] = 0.0;
  if (any_batch) {
    for (int64_t i = threadIdx.x; i < pn; i += blockDim.x) {
#pragma unroll
      for (int k = 0; k < 5; ++k) v[k] += a.part[k * st + p0 + i];
    }
    for (int64_t i = threadIdx.x; i < st; i += blockDim.x) {
#pragma unroll
      for (int k = 0; k < 5; ++k) v[5 + k] += a.part[k * st + i];
    }
    block_sum_n<10>(v, smem);
  } else {
    // group level only: the first wave sums the group's entries, the others wait for it
    if (threadIdx.x < 64) {
      for (int64_t i = threadIdx.x; i < pn; i += 64) {
#pragma unroll
        for (int k = 0; k < 5; ++k) v[k] += a.part[k * st + p0 + i];
      }
#pragma unroll
      for (int k = 0; k < 5; ++k) v[k] = wave_sum(v[k]);
      if (threadIdx.x == 0) {
#pragma unroll
        for (int k = 0; k < 5; ++k) smem[k] = v[k];
      }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 5; ++k) v[k] = smem[k];
    v[5] = v[0];
    if (has_mask && v[0] == 0.0) {  // nothing active in the group: is anything active at all?
      double c = 0.0;
      for (int64_t i = threadIdx.x; i < st; i += blockDim.x) c += a.part[i];
      v[5] = block_sum_d(c, smem + 8);
    }
  }
  if (has_mask && v[5] == 0.0) {  // nothing active: the input is returned unchanged
    for (int64_t i = lo + threadIdx.x; i < hi; i += blockDim.x) a.out[i] = a.x[i];
    return;
  }
  const NormParams np = norm_params(a, g, v);
  auto one = [&](float x, float m) -> float { return norm_one(np, x, m, has_mask); };
  for (int64_t i = lo + threadIdx.x; i < mid_lo; i += blockDim.x) a.out[i] = one(a.x[i], has_mask ? a.mask[i] : 1.0f);
  for (int64_t i = i0; i < mid_hi; i += 4 * step) {
    if (i != i0) fetch(i);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int64_t j = i + u * step;
      if (j >= mid_hi) break;
      f32x4 r;
#pragma unroll
      for (int e = 0; e < 4; ++e) r[e] = one(xv[u][e], mv[u][e]);
      *(f32x4*)(a.out + j) = r;
    }
  }
  for (int64_t i = mid_hi + threadIdx.x; i < hi; i += blockDim.x)
    if (i >= mid_lo) a.out[i] = one(a.x[i], has_mask ? a.mask[i] : 1.0f);
}

// The apply pass after the packed GAE (GaeArgs::seg_stats) over blocks of SEG_APPLY_ELEMS consecutive
// elements instead of (group, split): the grid depends on the number of elements alone, so nobody has
// to know the longest group (which meant waiting for the GPU), and uneven groups leave no block idle. A
// block finds the groups of its first and last element, requests its 16 elements per thread first, and
// then takes its groups (one or two) in turn. Groups as GaeArgs: token offsets or first sequences.
__global__ __launch_bounds__(NORM_THREADS) void norm_apply_seg_kernel(NormArgs a, GroupOffsets go) {
  __shared__ double smem[4 * 10];
  __shared__ int s_grp[2];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const bool has_mask = a.mask != nullptr;
  const int64_t lo = (int64_t)blockIdx.x * SEG_APPLY_ELEMS;
  const int64_t hi = lo + SEG_APPLY_ELEMS < a.n ? lo + SEG_APPLY_ELEMS : a.n;
  constexpr int U = SEG_APPLY_ELEMS / (4 * NORM_THREADS);
  f32x4 xv[U], mv[U], r[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int64_t j = lo + 4 * (tid + u * NORM_THREADS);
    xv[u] = f32x4{0.f, 0.f, 0.f, 0.f};
    mv[u] = f32x4{1.f, 1.f, 1.f, 1.f};
    if (j + 4 <= a.n) {
      xv[u] = *(const f32x4*)(a.x + j);
      if (has_mask) mv[u] = *(const f32x4*)(a.mask + j);
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (j + e < a.n) { xv[u][e] = a.x[j + e]; if (has_mask) mv[u][e] = a.mask[j + e]; }
    }
    r[u] = xv[u];
  }
  if (wave < 2) {
    GroupOffsets ends = go;
    ends.shift = 1;
    const int k = wave_count_le(ends, a.G, wave == 0 ? lo : hi - 1, lane);
    if (lane == 0) s_grp[wave] = k < a.G ? k : a.G - 1;
  }
  const bool any_batch = a.mean_level == LEVEL_BATCH || a.std_level == LEVEL_BATCH;
  const int64_t st = GAE_SEG_WAVES * a.part_slots;
  double v[10];
#pragma unroll
  for (int k = 0; k < 10; ++k) v[k] = 0.0;
  if (any_batch) {
    for (int64_t i = tid; i < st; i += NORM_THREADS) {
#pragma unroll
      for (int k = 0; k < 5; ++k) v[5 + k] += a.part[k * st + i];
    }
    block_sum_n<10>(v, smem);
  }
  __syncthreads();
  const int g_first = s_grp[0], g_last = s_grp[1];
  for (int g = g_first; g <= g_last; ++g) {
    const int64_t g0 = go[g], g1 = go[g + 1];
    __syncthreads();  // the previous group's readers are done
    if (wave == 0) {
      double w[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
      const int64_t p0 = GAE_SEG_WAVES * (g0 / a.part_tile + g);
      const int64_t pn = g1 > g0 ? GAE_SEG_WAVES * ((g1 - 1) / a.part_tile - g0 / a.part_tile + 1) : 0;
      for (int64_t i = lane; i < pn; i += 64) {
#pragma unroll
        for (int k = 0; k < 5; ++k) w[k] += a.part[k * st + p0 + i];
      }
#pragma unroll
      for (int k = 0; k < 5; ++k) w[k] = wave_sum(w[k]);
      if (lane == 0) {
#pragma unroll
        for (int k = 0; k < 5; ++k) smem[k] = w[k];
      }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 5; ++k) v[k] = smem[k];
    double active = any_batch ? v[5] : v[0];
    if (has_mask && !any_batch && active == 0.0) {  // nothing active in the group: is anything active at all?
      double c = 0.0;
      for (int64_t i = tid; i < st; i += NORM_THREADS) c += a.part[i];
      active = block_sum_d(c, smem + 8);
    }
    if (!any_batch) v[5] = active;
    if (has_mask && active == 0.0) continue;  // nothing active: the input is returned unchanged
    const NormParams np = norm_params(a, g, v);
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int64_t j = lo + 4 * (tid + u * NORM_THREADS) + e;
        if (j >= g0 && j < g1) r[u][e] = norm_one(np, xv[u][e], mv[u][e], has_mask);
      }
  }
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int64_t j = lo + 4 * (tid + u * NORM_THREADS);
    if (j + 4 <= a.n) *(f32x4*)(a.out + j) = r[u];
    else
#pragma unroll
      for (int e = 0; e < 4; ++e) if (j + e < a.n) a.out[j + e] = r[u][e];
  }
}

// Reward scores of a batch (actor.py:197-206): clip((reward + bias) * scaling, -clip, clip) and, with
// `normed`, their group or batch normalisation (no leave-one-out; groups of rows by a.goff), in one
// launch of one block: a batch has at most a few thousand rows, and the chain of tensor operations and
// the normalisation's two launches cost 5 us each. A wave takes whole groups. (Group levels alone:
// reward_score_groups_kernel.)
constexpr int SCORE_THREADS = 1024;
// As torch.clip: NaN stays, and the upper bound is the last word (a negative clip).
DEVI float shaped_reward(float reward, float bias, float scaling, float clip) {
  float x = (reward + bias) * scaling;
  x = x < -clip ? -clip : x;
  return x > clip ? clip : x;
}
__global__ __launch_bounds__(SCORE_THREADS) void reward_score_kernel(NormArgs a, float bias, float scaling, float clip,
                                                                     int normed) {
  constexpr int NW = SCORE_THREADS / 64;
  __shared__ double sm[NW][2];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  double b1 = 0.0, b4 = 0.0;
  for (int64_t i = tid; i < a.n; i += SCORE_THREADS) {
    const float x = shaped_reward(a.x[i], bias, scaling, clip);
    a.out[i] = x;
    b1 += (double)x;
    b4 += (double)x * (double)x;
  }
  if (!normed) return;
  double v[10];
#pragma unroll
  for (int k = 0; k < 10; ++k) v[k] = 0.0;
  b1 = wave_sum(b1);
  b4 = wave_sum(b4);
  if (lane == 0) { sm[wave][0] = b1; sm[wave][1] = b4; }
  __syncthreads();  // (also makes the block's stores to out visible to the block)
  for (int i = 0; i < NW; ++i) { v[6] += sm[i][0]; v[9] += sm[i][1]; }
  v[5] = v[7] = (double)a.n;
  v[8] = v[6];
  for (int g = wave; g < a.G; g += NW) {
    const int64_t g0 = a.goff[g], g1 = a.goff[g + 1];
    double s1 = 0.0, s4 = 0.0;
    for (int64_t i = g0 + lane; i < g1; i += 64) {
      const double x = (double)a.out[i];
      s1 += x;
      s4 += x * x;
    }
    s1 = wave_sum(s1);
    s4 = wave_sum(s4);
    v[0] = v[2] = (double)(g1 - g0);
    v[1] = v[3] = s1;
    v[4] = s4;
    const NormParams np = norm_params(a, g, v);
    for (int64_t i = g0 + lane; i < g1; i += 64) a.out[i] = norm_one(np, a.out[i], 1.f, false);
  }
}

// The same where no level is the batch: a wave of any block takes a whole group and needs nothing
// else, so the groups spread over the CUs (one block walks 64 groups of 16 rows in 10.2 us, latency of
// one group after the other; this 4.7). Rows behind the last group are only shaped.
__global__ __launch_bounds__(256) void reward_score_groups_kernel(NormArgs a, float bias, float scaling, float clip) {
  const int lane = threadIdx.x & 63, g = (int)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (g > a.G) return;
  auto shaped = [&](int64_t i) { return shaped_reward(a.x[i], bias, scaling, clip); };
  const int64_t g0 = a.goff[g], g1 = g < a.G ? a.goff[g + 1] : a.n;
  if (g == a.G) {
    for (int64_t i = g0 + lane; i < g1; i += 64) a.out[i] = shaped(i);
    return;
  }
  double v[10];
#pragma unroll
  for (int k = 0; k < 10; ++k) v[k] = 0.0;
  double s1 = 0.0, s4 = 0.0;
  for (int64_t i = g0 + lane; i < g1; i += 64) {
    const double x = (double)shaped(i);
    s1 += x;
    s4 += x * x;
  }
  s1 = wave_sum(s1);
  s4 = wave_sum(s4);
  v[0] = v[2] = (double)(g1 - g0);
  v[1] = v[3] = s1;
  v[4] = s4;
  const NormParams np = norm_params(a, g, v);
  for (int64_t i = g0 + lane; i < g1; i += 64) a.out[i] = norm_one(np, shaped(i), 1.f, false);
}

// pass 2: sum of squared masked deviations per (group, split)
__global__ __launch_bounds__(NORM_THREADS) void norm_stats2_kernel(NormArgs a) {
  __shared__ double smem[4];
  const int g = blockIdx.x, sp = blockIdx.y;
  const MeanCtx mc = make_mean_ctx(a, g, smem);
  int64_t lo, hi;
  split_range(a, g, sp, lo, hi);
  double ss = 0.0;
  const bool has_mask = a.mask != nullptr;
  for (int64_t i = lo + threadIdx.x; i < hi; i += blockDim.x) {
    const float x = a.x[i];
    const float m = has_mask ? a.mask[i] : 1.0f;
    const double mean = elem_mean(mc, x, m, has_mask);
    const double d = has_mask ? ((double)x * (double)m - mean * (double)m) : ((double)x - mean);
    ss += d * d;
  }
  ss = block_sum_d(ss, smem);
  if (threadIdx.x == 0) a.part[((int64_t)2 * a.G + g) * a.nsplit + sp] = ss;
}

// pass 3: normalise
__global__ __launch_bounds__(NORM_THREADS) void norm_apply_kernel(NormArgs a) {
  __shared__ double smem[4];
  const int g = blockIdx.x, sp = blockIdx.y;
  const bool has_mask = a.mask != nullptr;
  int64_t lo, hi;
  split_range(a, g, sp, lo, hi);
  if (has_mask) {
    const double total = batch_partial(a, 0, smem);
    if (total == 0.0) {  // nothing active: the input is returned unchanged
      for (int64_t i = lo + threadIdx.x; i < hi; i += blockDim.x) a.out[i] = a.x[i];
      return;
    }
  }
  const MeanCtx mc = make_mean_ctx(a, g, smem);
  // standard deviation
  double std_d = 1.0;
  double eps = a.eps;
  if (a.std_level == LEVEL_BATCH) {
    const double cnt = batch_partial(a, 0, smem);
    const double ss = batch_partial(a, 2, smem);
    if (a.unbiased) std_d = cnt <= 1.0 ? 1.0 : sqrt(ss / (cnt - 1.0));
    else std_d = cnt == 0.0 ? 1.0 : sqrt(ss / cnt);
  } else if (a.std_level == LEVEL_GROUP) {
    if (g == a.tail_group) std_d = 0.0;
    else if (a.grows[g] == 1 && a.unbiased) std_d = 1.0;
    else {
      const double cnt = group_partial(a, 0, g, smem);
      const double ss = group_partial(a, 2, g, smem);
      if (a.unbiased) std_d = cnt <= 1.0 ? 1.0 : sqrt(ss / (cnt - 1.0));
      else std_d = cnt == 0.0 ? 1.0 : sqrt(ss / cnt);
    }
    std_d = (double)(float)std_d;
  } else {
    eps = 0.0;
  }
  const bool mean64 = a.mean_level == LEVEL_BATCH, std64 = a.std_level == LEVEL_BATCH;
  for (int64_t i = lo + threadIdx.x; i < hi; i += blockDim.x) {
    const float x = a.x[i];
    const float m = has_mask ? a.mask[i] : 1.0f;
    const double mean = elem_mean(mc, x, m, has_mask);
    float r;
    if (mean64 || std64) {
      double c = mean64 ? ((double)x - mean) : (double)(x - (float)mean);
      if (has_mask) c = mean64 ? c * (double)m : (double)((float)c * m);
      const double den = std64 ? (std_d + eps) : (double)((float)std_d + (float)eps);
      r = (float)(c / den);
    } else {
      float c = x - (float)mean;
      if (has_mask) c = c * m;
      r = c / ((float)std_d + (float)eps);
    }
    a.out[i] = r;
  }
}

// masked_normalization (functional.py:16-53): one group, var = E[x^2] - E[x]^2 in fp64,
// (x*mask - mean) / (sqrt(var) + eps); the centred value is not re-masked.
__global__ __launch_bounds__(NORM_THREADS) void masked_norm_stats_kernel(const float* x,
                                                                          const float* mask,
                                                                          int64_t n, double* part) {
  __shared__ double smem[4];
  double cnt = 0.0, s = 0.0, s2 = 0.0;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x) {
    const double m = mask ? (double)mask[i] : 1.0;
    const double v = (double)x[i] * m;
    cnt += m; s += v; s2 += v * v;
  }
  cnt = block_sum_d(cnt, smem); s = block_sum_d(s, smem); s2 = block_sum_d(s2, smem);
  if (threadIdx.x == 0) {
    part[blockIdx.x] = cnt; part[gridDim.x + blockIdx.x] = s; part[2 * gridDim.x + blockIdx.x] = s2;
  }
}
__global__ __launch_bounds__(NORM_THREADS) void masked_norm_apply_kernel(
    const float* x, const float* mask, int64_t n, const double* part, int nparts, int unbiased,
    double eps, float* out) {
  __shared__ double smem[4];
  double cnt = 0.0, s = 0.0, s2 = 0.0;
  for (int i = threadIdx.x; i < nparts; i += blockDim.x) {
    cnt += part[i]; s += part[nparts + i]; s2 += part[2 * nparts + i];
  }
  cnt = block_sum_d(cnt, smem); s = block_sum_d(s, smem); s2 = block_sum_d(s2, smem);
  const double mean = s / cnt;
  double var = s2 / cnt - mean * mean;
  if (unbiased) var *= cnt / (cnt - 1.0);
  const double den = sqrt(var) + eps;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x) {
    const double v = (double)x[i] * (mask ? (double)mask[i] : 1.0);
    out[i] = (float)((v - mean) / den);
  }
}

// The same over each row of a [rows, cols] array (masked_normalization with dim = the trailing
// dimensions): one block per row, statistics then the apply pass over the row.
__global__ __launch_bounds__(NORM_THREADS) void masked_norm_rows_kernel(
    const float* x, const float* mask, int64_t cols, int unbiased, double eps, float* out) {
  __shared__ double smem[4];
  const float* xr = x + (int64_t)blockIdx.x * cols;
  const float* mr = mask ? mask + (int64_t)blockIdx.x * cols : nullptr;
  float* o = out + (int64_t)blockIdx.x * cols;
  double cnt = 0.0, s = 0.0, s2 = 0.0;
  for (int64_t i = threadIdx.x; i < cols; i += blockDim.x) {
    const double m = mr ? (double)mr[i] : 1.0;
    const double v = (double)xr[i] * m;
    cnt += m; s += v; s2 += v * v;
  }
  cnt = block_sum_d(cnt, smem); s = block_sum_d(s, smem); s2 = block_sum_d(s2, smem);
  const double mean = s / cnt;
  double var = s2 / cnt - mean * mean;
  if (unbiased) var *= cnt / (cnt - 1.0);
  const double den = sqrt(var) + eps;
  for (int64_t i = threadIdx.x; i < cols; i += blockDim.x) {
    const double v = (double)xr[i] * (mr ? (double)mr[i] : 1.0);
    o[i] = (float)((v - mean) / den);
  }
}

// ---------------------------------------------------------------------------------------
// Reward shaping in front of GAE (PPOActor.compute_advantages, areal/trainer/ppo/actor.py:224-283):
// one pass over a padded [bs, L] batch instead of some twenty elementwise tensor ops. One block
// per row; the row's sequence length (sum of the attention mask) first, then per token t:
//   lm[t]   = float(loss_mask[(t + 1) % L])                       (torch.roll(..., -1))
//   old[t]  = logp[(t + 1) % L] * lm[t]   (logp[t] * lm[t] when the log-probs are not rolled)
//   ref[t]  = ref_logp[t] * lm[t]         (0 when there is no reference policy)
//   kl[t]   = -kl_ctl * estimator(old[t] - ref[t])                (data.py:1662-1698)
//   gkl[t]  = kl[t], zero at t = seqlen - 1
//   out[t]  = reward_score at t = max(seqlen - 2, 0), else 0 (0 everywhere for a truncated
//             row when mask_no_eos_with_zero)
//   tot[t]  = gkl[t] + out[t]
// The arithmetic follows the reference's tensor ops in their order (this file is compiled
// without floating-point contraction). Index -1 of an empty row addresses the last slot, as
// Python indexing does.
// ---------------------------------------------------------------------------------------
struct PrepArgs {
  const uint8_t* loss_mask;  // [bs, L] nonzero = 1
  const uint8_t* attn_mask;  // [bs, L]
  const float* logp;         // [bs, L]
  float* ref_logp;           // [bs, L] or null; masked in place when ref_in_place
  const float* reward_score; // [bs]
  int64_t L;
  int roll_logp;             // 1: old = roll(logp, -1); 0: old = logp
  int estimator;             // 1, 2, 3
  int apply_clamp;
  int mask_no_eos_with_zero;
  int ref_in_place;
  float kl_ctl;
  float* lm_out;             // [bs, L]
  float* old_out;            // [bs, L]
  float* kl_out;             // [bs, L]  kl rewards before the end-of-sequence zero
  float* gkl_out;            // [bs, L] or null
  float* outcome_out;        // [bs, L] or null
  float* tot_out;            // [bs, L]
  int64_t* seqlens_out;      // [bs]
  uint8_t* no_eos_out;       // [bs]
};

DEVI void adv_prep_token(const PrepArgs& a, int estimator, float lm, float lp, float rf_in, bool has_ref, bool at_end,
                         bool at_out, float score, float neg_ctl, float& old, float& ref, float& kl,
                         float& gkl, float& oc) {
  old = lp * lm;
  ref = has_ref ? rf_in * lm : 0.f * lm;
  const float diff = old - ref;
  float est;
  if (estimator == 1) est = diff;
  else if (estimator == 2) est = diff * diff / 2.0f;
  else { const float neg = -diff; est = expf(neg) - 1.f - neg; }
  if (a.apply_clamp) est = est < -10.f ? -10.f : est > 10.f ? 10.f : est;  // (torch.clamp keeps NaN)
  kl = neg_ctl * est;
  gkl = at_end ? 0.f : kl;
  oc = at_out ? score : 0.f;
}

// Four tokens per thread and step, 16-byte loads and stores at whatever alignment the row has (the rolled
// neighbour of a group's last token is one extra scalar load), the row's last L % 4 tokens one by one. One token
// per thread and step, which rows of another length than a multiple of 16 used to take: a batch of
// 1000 x 8191 131 -> 111 us in all.
typedef u32x4 u32x4_any __attribute__((aligned(1)));
typedef uint32_t u32_any __attribute__((aligned(1)));
__global__ __launch_bounds__(NORM_THREADS) void adv_prep_kernel(PrepArgs a) {
  __shared__ double smem[4];
  const int64_t b = blockIdx.x, L = a.L;
  const uint8_t* am = a.attn_mask + b * L;
  const uint8_t* lmk = a.loss_mask + b * L;
  const float* lp = a.logp + b * L;
  float* rf = a.ref_logp ? a.ref_logp + b * L : nullptr;
  int cnt = 0;
  for (int64_t t = (int64_t)threadIdx.x * 16; t + 16 <= L; t += (int64_t)blockDim.x * 16) {
    const u32x4 w = *(const u32x4_any*)(am + t);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int k = 0; k < 4; ++k) cnt += ((w[i] >> (8 * k)) & 0xffu) ? 1 : 0;
  }
  if (threadIdx.x < (L & 15)) cnt += am[(L & ~(int64_t)15) + threadIdx.x] ? 1 : 0;
  const int64_t seqlen = (int64_t)block_sum_d((double)cnt, smem);
  const bool no_eos = seqlen == L;
  if (threadIdx.x == 0) { a.seqlens_out[b] = seqlen; a.no_eos_out[b] = no_eos ? 1 : 0; }
  const int64_t t_end = seqlen - 1 >= 0 ? seqlen - 1 : seqlen - 1 + L;  // rewards[b, seqlen - 1] = 0
  const int64_t t_out = seqlen - 2 > 0 ? seqlen - 2 : 0;                 // clip(seqlen - 2, min = 0)
  float score = a.reward_score[b];
  if (a.mask_no_eos_with_zero && no_eos) score = 0.f;
  const float neg_ctl = -a.kl_ctl;
  const bool has_ref = rf != nullptr;
  const int64_t L4 = L & ~(int64_t)3;
  for (int64_t t = (int64_t)threadIdx.x * 4; t < L4; t += (int64_t)blockDim.x * 4) {
    const int64_t tn = t + 4 < L ? t + 4 : 0;  // the roll's neighbour of the group's last token
    const uint32_t mw = *(const u32_any*)(lmk + t);
    const float lmv[4] = {((mw >> 8) & 0xffu) ? 1.f : 0.f, ((mw >> 16) & 0xffu) ? 1.f : 0.f,
                          (mw >> 24) ? 1.f : 0.f, lmk[tn] ? 1.f : 0.f};
    const f32x4 lv = *(const f32x4_any*)(lp + t);
    const float lpv[4] = {a.roll_logp ? lv[1] : lv[0], a.roll_logp ? lv[2] : lv[1],
                          a.roll_logp ? lv[3] : lv[2], a.roll_logp ? lp[tn] : lv[3]};
    f32x4 rv = {0.f, 0.f, 0.f, 0.f};
    if (has_ref) rv = *(const f32x4_any*)(rf + t);
    f32x4 o_lm, o_old, o_ref, o_kl, o_gkl, o_oc, o_tot;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float old, ref, kl, gkl, oc;
      adv_prep_token(a, a.estimator, lmv[i], lpv[i], rv[i], has_ref, t + i == t_end, t + i == t_out, score, neg_ctl,
                     old, ref, kl, gkl, oc);
      o_lm[i] = lmv[i]; o_old[i] = old; o_ref[i] = ref; o_kl[i] = kl; o_gkl[i] = gkl; o_oc[i] = oc;
      o_tot[i] = gkl + oc;
    }
    if (has_ref && a.ref_in_place) *(f32x4_any*)(rf + t) = o_ref;
    *(f32x4_any*)(a.lm_out + b * L + t) = o_lm;
    *(f32x4_any*)(a.old_out + b * L + t) = o_old;
    *(f32x4_any*)(a.kl_out + b * L + t) = o_kl;
    if (a.gkl_out) *(f32x4_any*)(a.gkl_out + b * L + t) = o_gkl;
    if (a.outcome_out) *(f32x4_any*)(a.outcome_out + b * L + t) = o_oc;
    *(f32x4_any*)(a.tot_out + b * L + t) = o_tot;
  }
  const int64_t t = L4 + threadIdx.x;
  if (t < L) {
    const int64_t tn = t + 1 < L ? t + 1 : 0;
    const float lm = lmk[tn] ? 1.f : 0.f;
    float old, ref, kl, gkl, oc;
    adv_prep_token(a, a.estimator, lm, a.roll_logp ? lp[tn] : lp[t], has_ref ? rf[t] : 0.f, has_ref, t == t_end,
                   t == t_out, score, neg_ctl, old, ref, kl, gkl, oc);
    if (has_ref && a.ref_in_place) rf[t] = ref;
    a.lm_out[b * L + t] = lm;
    a.old_out[b * L + t] = old;
    a.kl_out[b * L + t] = kl;
    if (a.gkl_out) a.gkl_out[b * L + t] = gkl;
    if (a.outcome_out) a.outcome_out[b * L + t] = oc;
    a.tot_out[b * L + t] = gkl + oc;
  }
}

// ---------------------------------------------------------------------------------------
// The whole of token-level advantages in front of their normalisation in one launch: a row's reward score
// (reward_score_groups_kernel's), adv_prep_kernel and gae_owned_kernel with the row sums, a block per row walking its
// tiles from the right, with the results of the three. Short batches are bound by latency (loads, sums, scan,
// each behind a barrier): the arrays that need neither the row's length nor its score are written while the
// last wave works the score out. Large ones are bound by HBM: the shaped rewards and the mask go from the shaping to
// the scan in registers instead of through memory.
// Kernels of the three calls and of this one: 64 x 1000 without a critic 17.5 -> 9.4 us; 1024 x 8192 with critic
// and reference 90 -> 66 us (42 B a slot in place of 50, 5.3 TB/s with inputs new to the caches). The rule for the
// rows' number and length is row_sums_fit. Reference and values with the non-temporal hint: 65 us there, but
// 20.2 against 18.0 at 400 x 3001, whose inputs are still in the last-level cache.
// A thread has the tokens of gae_row_tile.
// It loads the mask and the log-probs of its tokens from the tokens behind them (the roll), at whatever alignment
// that is; the one thread of a row whose tokens reach its end picks them one by one.
// ---------------------------------------------------------------------------------------
struct AdvGaeArgs {
  PrepArgs p;                 // reward_score: the scores, with score_mode 0
  GaeArgs g;                  // rewards and mask unused
  int score_mode;             // 1: scores are shaped here, 2: and normalised within groups
  NormArgs score;             // x = raw rewards [bs], groups of rows
  float bias, scaling, clip;
  // NORM: normalisation of the advantages within groups of rows (goff in elements), see adv_normalise_row
  NormArgs norm;
  uint64_t *sums, *flags, *left;  // [bs][4] and twice [bs] in the workspace
  uint64_t call;              // a number no other call has
  unsigned wait_ticks;        // of the 100 MHz clock
};

// ---- Normalisation in the launch that made the advantages: a row's block keeps them in LDS, hands the row's sums to
// the blocks of its group and waits for theirs, up to ADV_GROUP_ROWS rows. The batch's advantages then go to memory once
// instead of being written, read back with the mask and written again by a launch of its own (42 against 54 B a
// slot, and 5 us less for a small batch).
// No wait is unbounded: the blocks of a group lie next to each other in the grid, but nobody promises that they
// are on the chip together. A block whose time is up stores its row as it is and leaves a note (`left`); it, or any
// block of the group that finds all sums, then takes the note (one of them, by compare and swap) and normalises that row
// from memory. Leaving a note is followed by another look at the sums, publishing one's sums precedes the look for notes:
// of the block that leaves one and the last of the group to publish, one sees the other (the order stands at leave_note).
constexpr int ADV_GROUP_ROWS = 64;                   // one lane per row
constexpr int ADV_NORM_TILES = 4;                    // of a row, 8 mask bits each
struct RowGroup { int g, first, rows; };  // group of a row: its first row and their number
DEVI RowGroup row_group(const NormArgs& n, int64_t row, int64_t L) {  // by a whole wave; row: the row's first element
  const int g = wave_count_le(n.goff + 1, n.G, row, threadIdx.x & 63);
  const int64_t e0 = n.goff[g], e1 = n.goff[g + 1];
  return RowGroup{g, (int)(e0 / L), (int)((e1 - e0) / L)};
}
// Row b from LDS (x, `bits`: the mask of the thread's tokens, 8 a tile), after its scan; s: its sums.
DEVI void adv_normalise_row(const AdvGaeArgs& a, int64_t b, const RowGroup& rg, const float* x, uint32_t bits,
                            const double (&s)[3]) {
  __shared__ double s_sum[3];
  __shared__ int s_flag;
  __shared__ uint64_t s_todo;
  const int tid = threadIdx.x, L = (int)a.p.L;
  float* const adv = a.g.adv + b * L;
  auto of_tiles = [&](auto&& f) {
    for (int tile = (L - 1) / GAE_TILE; tile >= 0; --tile) {
      const int t0 = row_tile_token(tile);
#pragma unroll
      for (int q = 0; q < ROW_QUADS; ++q)
        row_store<false>(adv, t0, L, q, f(*(const f32x4*)(x + t0 + q * WAVE_QUADS), bits >> (8 * tile + QUAD * q)));
    }
  };
  if (tid == 0) publish_sums(a.sums + 4 * b, a.flags + b, a.call, s);
  uint64_t todo = 0;  // (first wave) rows of the group whose blocks have left
  auto gather = [&](unsigned ticks) {
    if (tid < 64) {
      double v[3];
      const bool all = gather_sums<4>(a.sums + 4 * (int64_t)rg.first, a.flags + rg.first, rg.rows, a.call, wall_clock64() + ticks, v);
      if (tid == 0) {
        s_flag = all ? 1 : 0;
#pragma unroll
        for (int k = 0; k < 3; ++k) s_sum[k] = v[k];
      }
      if (all) {
        published_before_notes();
        todo = __builtin_amdgcn_ballot_w64(tid < rg.rows && note_left(a.left + rg.first + tid, a.call));
      }
    }
    __syncthreads();
    return s_flag != 0;
  };
  if (!gather(a.wait_ticks)) {
    of_tiles([&](const f32x4& w, uint32_t) { return w; });
    __threadfence();
    __syncthreads();
    if (tid == 0) leave_note(a.left + b, a.call);
    if (!gather(0)) return;
    // (its own note among the others' now)
  } else {
    double v[10];
    v[0] = v[2] = s_sum[0]; v[1] = v[3] = s_sum[1]; v[4] = s_sum[2];
#pragma unroll
    for (int k = 5; k < 10; ++k) v[k] = 0.0;
    const NormParams np = norm_params(a.norm, rg.g, v, [&] { return rg.rows; });
    of_tiles([&](const f32x4& w, uint32_t m) {
      f32x4 r;
#pragma unroll
      for (int e = 0; e < QUAD; ++e) r[e] = norm_one(np, w[e], (m >> e) & 1u ? 1.f : 0.f, true);
      return r;
    });
  }
  if (tid == 0) s_todo = todo;
  __syncthreads();
  for (uint64_t rest = s_todo; rest != 0; rest &= rest - 1) {
    const int64_t r = rg.first + __builtin_ctzll(rest);
    __syncthreads();
    if (tid == 0) s_flag = take_note(a.left + r, a.call) ? 1 : 0;
    __syncthreads();
    if (s_flag == 0) continue;  // somebody else's
    __threadfence();
    double v[10];
    v[0] = v[2] = s_sum[0]; v[1] = v[3] = s_sum[1]; v[4] = s_sum[2];
#pragma unroll
    for (int k = 5; k < 10; ++k) v[k] = 0.0;
    const NormParams np = norm_params(a.norm, rg.g, v, [&] { return rg.rows; });
    float* const to = a.g.adv + r * L;
    const float* const m = a.p.lm_out + r * L;
    for (int t = tid; t < L; t += GAE_THREADS) to[t] = norm_one(np, to[t], m[t], true);
  }
}

// Score of row b, by a whole wave. The sums run in reward_score_groups_kernel's order.
DEVI float row_score(const AdvGaeArgs& a, int64_t b) {
  if (a.score_mode == 0) return a.p.reward_score[b];
  const NormArgs& n = a.score;
  auto shaped = [&](int64_t i) { return shaped_reward(n.x[i], a.bias, a.scaling, a.clip); };
  const int lane = threadIdx.x & 63;
  if (a.score_mode == 1 || b >= n.goff[n.G]) return shaped(b);
  int lo = 0, hi = n.G;  // goff[lo] <= b < goff[hi]
  while (hi - lo > 1) {
    const int step = (hi - lo + 63) >> 6, i = lo + lane * step;
    const uint64_t le = __builtin_amdgcn_ballot_w64(i < hi && n.goff[i] <= b);
    lo += (__builtin_popcountll(le) - 1) * step;
    hi = lo + step < hi ? lo + step : hi;
  }
  const int64_t g0 = n.goff[lo], g1 = n.goff[lo + 1];
  double v[10], s1 = 0.0, s4 = 0.0;
#pragma unroll
  for (int k = 0; k < 10; ++k) v[k] = 0.0;
  for (int64_t i = g0 + lane; i < g1; i += 64) {
    const double x = (double)shaped(i);
    s1 += x;
    s4 += x * x;
  }
  s1 = wave_sum(s1);
  s4 = wave_sum(s4);
  v[0] = v[2] = (double)(g1 - g0);
  v[1] = v[3] = s1;
  v[4] = s4;
  return norm_one(norm_params(n, lo, v), shaped(b), 1.f, false);
}


// Inputs of a thread's two quads from t0 and t0 + WAVE_QUADS of a row on: rolled mask bytes and log-probs, reference,
// values. END: they may reach the end of the row.
struct PrepItems {
  uint32_t m[ROW_QUADS];
  float lp[GAE_ITEMS], rf[GAE_ITEMS], v[GAE_ITEMS];
};
template <bool END>
DEVI void prep_load(const AdvGaeArgs& a, int64_t row, int t0, PrepItems& x) {
  const int L = (int)a.p.L, roll = a.p.roll_logp ? 1 : 0;
  const uint8_t* const lm = a.p.loss_mask + row;
  const float *const lp = a.p.logp + row, *const rf = a.p.ref_logp != nullptr ? a.p.ref_logp + row : nullptr,
              *const v = a.g.values != nullptr ? a.g.values + row : nullptr;
#pragma unroll
  for (int i = 0; i < GAE_ITEMS; ++i) x.lp[i] = x.rf[i] = x.v[i] = 0.f;
#pragma unroll
  for (int q = 0; q < ROW_QUADS; ++q) {
    const int tq = t0 + q * WAVE_QUADS;
    x.m[q] = 0u;
    if (!END || tq + QUAD < L) {
      x.m[q] = *(const u32_any*)(lm + tq + 1);
      const f32x4 w = *(const f32x4_any*)(lp + tq + roll);
#pragma unroll
      for (int e = 0; e < QUAD; ++e) x.lp[QUAD * q + e] = w[e];
      if (rf != nullptr) {
        const f32x4 u = *(const f32x4_any*)(rf + tq);
#pragma unroll
        for (int e = 0; e < QUAD; ++e) x.rf[QUAD * q + e] = u[e];
      }
      if (v != nullptr) {
        const f32x4 u = *(const f32x4_any*)(v + tq);
#pragma unroll
        for (int e = 0; e < QUAD; ++e) x.v[QUAD * q + e] = u[e];
      }
    } else {
      // the end of the row: its last token's neighbour is its first
#pragma unroll
      for (int e = 0; e < QUAD; ++e) {
        const int t = tq + e, tn = t + 1 < L ? t + 1 : 0;
        if (t >= L) break;
        x.m[q] |= (uint32_t)lm[tn] << (8 * e);
        x.lp[QUAD * q + e] = lp[roll ? tn : t];
        if (rf != nullptr) x.rf[QUAD * q + e] = rf[t];
        if (v != nullptr) x.v[QUAD * q + e] = v[t];
      }
    }
  }
}

template <int EST, bool ONE_TILE, bool NORM>
__global__ __launch_bounds__(GAE_THREADS, 4) void adv_gae_kernel(AdvGaeArgs a) {
  extern __shared__ __attribute__((aligned(16))) float row_adv[];  // NORM: whole tiles
  __shared__ RowGroup s_group;
  __shared__ RowMaps maps;
  __shared__ double s_rs[4 * 5];
  __shared__ float s_score;
  const PrepArgs& p = a.p;
  const int tid = threadIdx.x, L = (int)p.L;
  const int64_t b = blockIdx.x, row = b * L;
  int tile = ONE_TILE ? 0 : (L - 1) / GAE_TILE;
  int t0 = row_tile_token(tile);
  PrepItems x;
  prep_load<true>(a, row, t0, x);
  int cnt = 0;
  const uint8_t* am = p.attn_mask + row;
  for (int t = tid * 8; t + 8 <= L; t += GAE_TILE) {
    const u32x2 w = *(const u32x2_any*)(am + t);
#pragma unroll
    for (int k = 0; k < 8; ++k) cnt += ((w[k >> 2] >> (8 * (k & 3))) & 0xffu) ? 1 : 0;
  }
  if (tid < (L & 7)) cnt += am[(L & ~7) + tid] ? 1 : 0;
  if (tid >= GAE_THREADS - 64) {
    const float sc = row_score(a, b);
    if (tid == GAE_THREADS - 1) s_score = sc;
  }
  if (NORM && tid < 64) {
    const RowGroup rg = row_group(a.norm, row, L);
    if (tid == 0) s_group = rg;
  }
  const float neg_ctl = -p.kl_ctl;
  const bool has_ref = p.ref_logp != nullptr;
  double A0 = 0.0, nv0 = 0.0, rs[5] = {0.0};  // state entering the tile from its right; sums of the row
  uint32_t bits = 0;
  int t_zero = 0, t_out = 0, no_eos = 0;
  float score = 0.f;
  for (bool first = true;; first = false) {
    float rw[GAE_ITEMS];  // first the KL rewards
    const ByteMask mask_of{x.m};
#pragma unroll
    for (int q = 0; q < ROW_QUADS; ++q) {
      f32x4 o_lm, o_old, o_ref, o_kl;
#pragma unroll
      for (int e = 0; e < QUAD; ++e) {
        const int i = QUAD * q + e;
        const float lm = mask_of(i);
        float old, ref, kl, gkl, oc;
        adv_prep_token(p, EST, lm, x.lp[i], x.rf[i], has_ref, false, false, 0.f, neg_ctl, old, ref, kl, gkl, oc);
        o_lm[e] = lm; o_old[e] = old; o_ref[e] = ref; o_kl[e] = kl;
        rw[i] = kl;
      }
      if (has_ref && p.ref_in_place) row_store<false>(p.ref_logp + row, t0, L, q, o_ref);
      row_store<false>(p.lm_out + row, t0, L, q, o_lm);
      row_store<true>(p.old_out + row, t0, L, q, o_old);
      row_store<true>(p.kl_out + row, t0, L, q, o_kl);
    }
    if (first) {  // (in scalar registers from here on)
      const int seqlen = __builtin_amdgcn_readfirstlane((int)block_sum_d((double)cnt, s_rs));
      no_eos = seqlen == L ? 1 : 0;
      if (tid == 0) { p.seqlens_out[b] = seqlen; p.no_eos_out[b] = (uint8_t)no_eos; }
      t_zero = seqlen > 0 ? seqlen - 1 : L - 1;
      t_out = seqlen > 2 ? seqlen - 2 : 0;
      const float sc = s_score;
      score = __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, sc)));
      if (p.mask_no_eos_with_zero && no_eos) score = 0.f;
    }
#pragma unroll
    for (int q = 0; q < ROW_QUADS; ++q) {
      f32x4 o_tot;
#pragma unroll
      for (int e = 0; e < QUAD; ++e) {
        const int t = t0 + q * WAVE_QUADS + e;
        const float gkl = t == t_zero ? 0.f : rw[QUAD * q + e], oc = t == t_out ? score : 0.f;
        o_tot[e] = gkl + oc;
        rw[QUAD * q + e] = o_tot[e];
      }
      row_store<false>(p.tot_out + row, t0, L, q, o_tot);
    }
    if constexpr (NORM) {
#pragma unroll
      for (int i = 0; i < GAE_ITEMS; ++i) bits |= (mask_of(i) != 0.f ? 1u : 0u) << (8 * tile + i);
    }
    gae_row_tile<true, true>(
        a.g.discount, a.g.lam, tile, t0, L, no_eos != 0, rw, x.v, mask_of, maps, A0, nv0, rs,
        [&](int q, const f32x4& w) {
          if constexpr (NORM) *(f32x4*)(row_adv + t0 + q * WAVE_QUADS) = w;
          else row_store<false>(a.g.adv + row, t0, L, q, w);
        },
        a.g.ret + row);
    if (ONE_TILE || --tile < 0) break;
    t0 -= GAE_TILE;
    prep_load<false>(a, row, t0, x);
  }
  // (the mask is 0 or 1)
  double s[3] = {rs[0], rs[1], rs[4]};
  block_sum_n<3>(s, s_rs);
  if constexpr (NORM) {
    adv_normalise_row(a, b, s_group, row_adv, bits, s);
  } else if (tid == 0) {
    double* const to = a.g.row_stats + b;
    const int64_t st = a.g.n_seqs;
    to[0] = to[2 * st] = s[0];
    to[st] = to[3 * st] = s[1];
    to[4 * st] = s[2];
  }
}

// ---------------------------------------------------------------------------------------
// Turn-level GAE (areal/trainer/ppo/gae.py:82-163): every generated turn is one timestep.
// One block per padded row. Active tokens carry non-decreasing turn ids (checked; a violation
// sets *status), so a turn starts at the first active token whose id exceeds every active id on
// its left. Pass 1 compacts the turns: start position's value, and the fp64 prefix sum of the
// active rewards taken just before the start (turn reward = difference of consecutive
// prefixes). Thread 0 then runs the recurrence over the compact turns right to left, and pass
// 2 hands every token its turn's advantage and return.
// Per row workspace: prefix [L+1] double, value/adv/ret [L] float each; a row of at most TURN_LDS turns (a
// conversation has tens) keeps them in LDS.
// A row is bound by latency: loads, two scans behind barriers per tile of the row, the recurrence. Blocks of up to
// 1024 threads therefore, so that a row is one or two tiles, 16-byte accesses, and the recurrence from LDS (from global
// memory it waited for a load per turn): 128 x 8192 53 -> 21 us, 512 x 4096 36 -> 19,
// 1024 x 8192 88 -> 58, 64 x 1000 9.0 -> 6.2.
// ---------------------------------------------------------------------------------------
constexpr int TURN_THREADS = 256;
constexpr int TURN_ITEMS = 4;
constexpr int TURN_LDS = 512;
typedef int i32x4_any __attribute__((ext_vector_type(4), aligned(4)));

struct TurnArgs {
  const float* rewards;
  const float* values;
  const float* mask;       // float loss mask, nonzero = active
  const int32_t* turn_ids;
  const uint8_t* no_eos;   // [bs] or null
  const float* lam_seq;    // [bs] or null
  int64_t bs, L;
  float discount, lam;
  float* adv;
  float* ret;
  double* ws_prefix;       // [bs][L + 1]
  float* ws_val;           // [bs][L]
  float* ws_adv;           // [bs][L]
  float* ws_ret;           // [bs][L]
  int* status;             // bit 0: negative id, bit 1: id >= L, bit 2: ids go backwards
  int roll;                // the ids are those of the token before (next-token convention): id[t + 1], -1 at the end
  const float* addend;     // [bs][L] or null: added to the advantages
};

struct TurnCarry { int count; int maxid; double sum; };

// Exclusive scan over the block of (start count, running max id, reward sum), chunk carry
// included. smem: an entry per wave of each.
template <int THREADS>
DEVI TurnCarry turn_block_exclusive(int cnt, int mx, double sm, const TurnCarry& carry, int* s_cnt,
                                    int* s_max, double* s_sum, TurnCarry& chunk_total) {
  // s_cnt / s_max / s_sum: one entry per wave. Scans inside a wave through DPP, the waves' totals
  // through LDS: two barriers.
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int ic = wave_inclusive_scan(cnt, 0, [](int a, int b) { return a + b; });
  const int im = wave_inclusive_scan(mx, -1, [](int a, int b) { return a > b ? a : b; });
  const double is = wave_inclusive_scan(sm, 0.0, [](double a, double b) { return a + b; });
  __syncthreads();  // the previous chunk's readers are done
  if (lane == 63) { s_cnt[w] = ic; s_max[w] = im; s_sum[w] = is; }
  __syncthreads();
  TurnCarry ex = carry;
  for (int i = 0; i < w; ++i) {
    ex.count += s_cnt[i];
    ex.maxid = ex.maxid > s_max[i] ? ex.maxid : s_max[i];
    ex.sum += s_sum[i];
  }
  chunk_total = carry;
#pragma unroll
  for (int i = 0; i < THREADS / 64; ++i) {
    chunk_total.count += s_cnt[i];
    chunk_total.maxid = chunk_total.maxid > s_max[i] ? chunk_total.maxid : s_max[i];
    chunk_total.sum += s_sum[i];
  }
  // the lanes before this one in its wave
  const int pc = wave_shift_up(ic, 0), pm = wave_shift_up(im, -1);
  const double ps = wave_shift_up(is, 0.0);
  ex.count += pc;
  ex.maxid = ex.maxid > pm ? ex.maxid : pm;
  ex.sum += ps;
  return ex;
}

template <int THREADS>
__global__ __launch_bounds__(THREADS) void turn_gae_kernel(TurnArgs a) {
  __shared__ int s_cnt[THREADS / 64], s_max[THREADS / 64];
  __shared__ double s_sum[THREADS / 64];
  __shared__ double s_prefix[TURN_LDS + 1];
  __shared__ float s_val[TURN_LDS], s_adv[TURN_LDS], s_ret[TURN_LDS];
  constexpr int TILE = THREADS * TURN_ITEMS;
  const int tid = threadIdx.x;
  const int64_t row = blockIdx.x, L = a.L;
  const float* rw = a.rewards + row * L;
  const float* vl = a.values != nullptr ? a.values + row * L : nullptr;  // (no critic: zero)
  const float* ms = a.mask + row * L;
  const float* add = a.addend != nullptr ? a.addend + row * L : nullptr;
  const int32_t* ids_row = a.turn_ids + row * L;
  double* prefix = a.ws_prefix + row * (L + 1);
  float* tval = a.ws_val + row * L;
  float* tadv = a.ws_adv + row * L;
  float* tret = a.ws_ret + row * L;
  auto load4 = [&](const float* from, int64_t t0, float (&x)[TURN_ITEMS]) {
    if (from != nullptr && t0 + TURN_ITEMS <= L) {
      const f32x4 w = *(const f32x4_any*)(from + t0);
#pragma unroll
      for (int i = 0; i < TURN_ITEMS; ++i) x[i] = w[i];
    } else {
#pragma unroll
      for (int i = 0; i < TURN_ITEMS; ++i) x[i] = from != nullptr && t0 + i < L ? from[t0 + i] : 0.f;
    }
  };
  int bad = 0;

  // A tile's tokens of this thread: mask, active ones and turn starts among them (bits), turns that started
  // before the first of them; with SUMS also their active rewards and the sum of those before them.
  float m[TURN_ITEMS], r[TURN_ITEMS];
  unsigned act, start;
  int k0;
  double sum0;
  auto scan_tile = [&](auto sums, int64_t t0, TurnCarry& carry) {
    constexpr bool SUMS = decltype(sums)::value;
    int ids[TURN_ITEMS];
    load4(ms, t0, m);
    if (t0 + TURN_ITEMS < L) {
      const i32x4_any w = *(const i32x4_any*)(ids_row + t0 + (a.roll ? 1 : 0));
#pragma unroll
      for (int i = 0; i < TURN_ITEMS; ++i) ids[i] = w[i];
    } else {
#pragma unroll
      for (int i = 0; i < TURN_ITEMS; ++i) {
        const int64_t t = t0 + i + (a.roll ? 1 : 0);
        ids[i] = t < L ? ids_row[t] : -1;
      }
    }
    if (SUMS) load4(rw, t0, r);
    int mx = -1;
    double sm = 0.0;
    act = start = 0;
#pragma unroll
    for (int i = 0; i < TURN_ITEMS; ++i) {
      const bool on = m[i] != 0.0f;
      if (SUMS) r[i] = on ? r[i] : 0.0f;
      if (!on) continue;
      act |= 1u << i;
      if (ids[i] < 0) bad |= 1;
      if ((int64_t)ids[i] >= L) bad |= 2;
      mx = mx > ids[i] ? mx : ids[i];
      if (SUMS) sm += (double)r[i];
    }
    // the number of starts in a thread depends on the maximum to its left, so scan the maximum
    // and the reward sums first, then count starts, then scan the counts
    TurnCarry tot1, tot2;
    const TurnCarry ex1 = turn_block_exclusive<THREADS>(0, mx, sm, carry, s_cnt, s_max, s_sum, tot1);
    int run_max = ex1.maxid;
#pragma unroll
    for (int i = 0; i < TURN_ITEMS; ++i) {
      if (!((act >> i) & 1u)) continue;
      if (ids[i] > run_max) start |= 1u << i;
      if (ids[i] < run_max) bad |= 4;
      run_max = run_max > ids[i] ? run_max : ids[i];
    }
    const TurnCarry ex2 = turn_block_exclusive<THREADS>(__popc(start), -1, 0.0, TurnCarry{carry.count, -1, 0.0}, s_cnt,
                                                        s_max, s_sum, tot2);
    k0 = ex2.count;
    sum0 = ex1.sum;
    carry = TurnCarry{tot2.count, tot1.maxid, tot1.sum};
  };

  // ---- pass 1: compact the turns
  TurnCarry carry{0, -1, 0.0};
  for (int64_t base = 0; base < L; base += TILE) {
    const int64_t t0 = base + (int64_t)tid * TURN_ITEMS;
    scan_tile(std::true_type{}, t0, carry);
    int k = k0;
    double run_sum = sum0;
#pragma unroll
    for (int i = 0; i < TURN_ITEMS; ++i) {
      if ((start >> i) & 1u) {
        const float v = vl != nullptr ? vl[t0 + i] : 0.f;  // the turn's state value: value at its first token
        if (k < TURN_LDS) { s_prefix[k] = run_sum; s_val[k] = v; }
        prefix[k] = run_sum;  // active rewards strictly before this turn
        tval[k] = v;
        ++k;
      }
      run_sum += (double)r[i];
    }
  }
  const int K = carry.count;  // (the same in every thread)
  if (tid == 0) {
    prefix[K] = carry.sum;
    if (K <= TURN_LDS) s_prefix[K] = carry.sum;
  }
  if (bad) atomicOr(a.status, bad);
  bad = 0;
  __syncthreads();
  __threadfence_block();

  // ---- recurrence over the turns, right to left (gae.py:139-150)
  const bool in_lds = K <= TURN_LDS;
  if (tid == 0) {
    const float gam = a.discount;
    const float lam = a.lam_seq ? a.lam_seq[row] : a.lam;
    const float c = gam * lam;
    auto recur = [&](const double* prefix, const float* tval, float* tadv, float* tret) {
      float nextv = (a.no_eos && a.no_eos[row]) ? (vl != nullptr ? vl[L - 1] : 0.f) : 0.0f;
      float last = 0.0f;
      for (int k = K - 1; k >= 0; --k) {
        const float R = (float)(prefix[k + 1] - prefix[k]);
        const float V = tval[k];
        const float delta = (R + gam * nextv) - V;
        const float g = delta + c * last;
        tadv[k] = g;
        tret[k] = g + V;
        nextv = V;
        last = g;
      }
    };
    if (in_lds) recur(s_prefix, s_val, s_adv, s_ret);
    else recur(prefix, tval, tadv, tret);
  }
  __syncthreads();
  __threadfence_block();

  // ---- pass 2: every token takes the result of its turn (gae.py:152-157); a row of one tile still has what
  // pass 1 found
  TurnCarry carry2{0, -1, 0.0};
  for (int64_t base = 0; base < L; base += TILE) {
    const int64_t t0 = base + (int64_t)tid * TURN_ITEMS;
    float v[TURN_ITEMS], ad[TURN_ITEMS];
    load4(vl, t0, v);
    load4(add, t0, ad);
    if (L > TILE) scan_tile(std::false_type{}, t0, carry2);
    int k = k0;  // turns started strictly before this thread's first token
    f32x4 o_adv, o_ret;
#pragma unroll
    for (int i = 0; i < TURN_ITEMS; ++i) {
      if ((start >> i) & 1u) ++k;
      float adv = 0.0f, ret = v[i];
      if (((act >> i) & 1u) && k > 0) {
        const float mm = m[i];
        adv = (in_lds ? s_adv[k - 1] : tadv[k - 1]) * mm;
        ret = (in_lds ? s_ret[k - 1] : tret[k - 1]) * mm + ret * (1.0f - mm);
      }
      o_adv[i] = add != nullptr ? adv + ad[i] : adv;
      o_ret[i] = ret;
    }
    if (t0 + TURN_ITEMS <= L) {
      *(f32x4_any*)(a.adv + row * L + t0) = o_adv;
      *(f32x4_any*)(a.ret + row * L + t0) = o_ret;
    } else {
#pragma unroll
      for (int i = 0; i < TURN_ITEMS - 1; ++i)
        if (t0 + i < L) { a.adv[row * L + t0 + i] = o_adv[i]; a.ret[row * L + t0 + i] = o_ret[i]; }
    }
  }
}

// Per-row lengths for the per-sample lambda functions (_build_gae_lambda_context,
// areal/trainer/ppo/gae.py:166-205): number of active tokens, and number of distinct turn ids
// among them (= turn starts, ids being non-decreasing over the active tokens; violations are
// reported through *status as in turn_gae_kernel). turn_ids may be null (turn count 0).
__global__ __launch_bounds__(TURN_THREADS) void gae_context_kernel(const float* mask,
                                                                   const int32_t* turn_ids, int64_t L,
                                                                   int64_t* token_len,
                                                                   int64_t* turn_cnt, int* status) {
  __shared__ int s_cnt[TURN_THREADS];
  __shared__ int s_max[TURN_THREADS];
  __shared__ double s_sum[TURN_THREADS];
  const int tid = threadIdx.x;
  const int64_t row = blockIdx.x;
  const float* ms = mask + row * L;
  const int32_t* id = turn_ids ? turn_ids + row * L : nullptr;
  int bad = 0;
  TurnCarry carry{0, -1, 0.0};
  int64_t starts = 0;
  for (int64_t base = 0; base < L; base += TURN_THREADS * TURN_ITEMS) {
    const int64_t t0 = base + (int64_t)tid * TURN_ITEMS;
    int ids[TURN_ITEMS]; bool act[TURN_ITEMS];
    int mx = -1, nact = 0;
#pragma unroll
    for (int i = 0; i < TURN_ITEMS; ++i) {
      const int64_t t = t0 + i;
      act[i] = t < L && ms[t] != 0.0f;
      ids[i] = (act[i] && id) ? id[t] : -1;
      nact += act[i];
      if (act[i] && id) {
        if (ids[i] < 0) bad |= 1;
        if ((int64_t)ids[i] >= L) bad |= 2;
        mx = mx > ids[i] ? mx : ids[i];
      }
    }
    TurnCarry tot;
    // count: active tokens; max: running turn id; sum unused
    const TurnCarry ex = turn_block_exclusive<TURN_THREADS>(nact, mx, 0.0, carry, s_cnt, s_max, s_sum, tot);
    int run_max = ex.maxid;
#pragma unroll
    for (int i = 0; i < TURN_ITEMS; ++i) {
      if (!act[i] || !id) continue;
      if (ids[i] > run_max) ++starts;
      if (ids[i] < run_max) bad |= 4;
      run_max = run_max > ids[i] ? run_max : ids[i];
    }
    carry = tot;
  }
  // total of the per-thread start counts
  __syncthreads();
  s_cnt[tid] = (int)starts;
  __syncthreads();
  if (tid == 0) {
    long long tot = 0;
    for (int i = 0; i < TURN_THREADS; ++i) tot += s_cnt[i];
    token_len[row] = carry.count;
    turn_cnt[row] = tot;
  }
  if (bad) atomicOr(status, bad);
}

// gae_owned_kernel's instance for the batch (STATS needs block = row)
template <bool STATS>
void launch_gae_owned(const GaeArgs& g, int64_t grid, hipStream_t stream) {
  const dim3 gr((unsigned)grid), bl(GAE_THREADS);
  if (g.block_per_seq) {
    if (g.lam_seq != nullptr) hipLaunchKernelGGL((gae_owned_kernel<STATS, true, true>), gr, bl, 0, stream, g);
    else hipLaunchKernelGGL((gae_owned_kernel<STATS, true, false>), gr, bl, 0, stream, g);
  } else if constexpr (!STATS) {
    if (g.lam_seq != nullptr) hipLaunchKernelGGL((gae_owned_kernel<false, false, true>), gr, bl, 0, stream, g);
    else hipLaunchKernelGGL((gae_owned_kernel<false, false, false>), gr, bl, 0, stream, g);
  }
}

uint64_t call_seed() noexcept {  // (random_device may throw, and no exception may leave a C entry)
  try {
    return ((uint64_t)std::random_device{}() << 32) ^ std::random_device{}();
  } catch (...) {
    return (uint64_t)std::chrono::steady_clock::now().time_since_epoch().count() * 0x9e3779b97f4a7c15ull;
  }
}
// A number no other call has, and no memory by chance.
uint64_t next_call_number() {
  static const uint64_t seed = call_seed();
  static std::atomic<uint64_t> calls{0};
  uint64_t z = seed + (calls.fetch_add(1, std::memory_order_relaxed) + 1) * 0x9e3779b97f4a7c15ull;  // splitmix64
  z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
  z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
  return z ^ (z >> 31);
}

// Ticks of the 100 MHz clock that a block waits for its group.
unsigned group_wait_ticks(int us) { return 100u * (unsigned)(us < 0 ? 200 : std::min(us, 1000)); }

// Whether the row sums ride in the scan of padded rows.
bool row_sums_fit(int64_t n_seqs, int64_t uniform_len) {
  if (uniform_len > 64 * (int64_t)GAE_TILE || n_seqs > (1 << 30)) return false;
  // A block per row: rows shorter than a tile leave lanes idle. While all blocks are resident (4 a CU) that
  // is cheaper than a launch of its own for the sums (all kernels of an advantage computation, rows x
  // slots: 64 x 1000 21.4 against 24.4 us, 1024 x 1000 33.4 against 35.4, 1024 x 64 20.8 against 21.3), with
  // many more short rows it is not, one launch for everything included (4096 x 256 43.6 against 35.9, 4096 x 512
  // 47.6 against 42.5, 8192 x 512 83.0 against 61.3). Rows of nearly a tile fill their block whatever their number.
  return uniform_len >= GAE_TILE - GAE_TILE / 8 || n_seqs <= 1024;
}

// Whether the normalisation of the scores rides in front of it (score_mode 2 of adv_gae_kernel): every row's last
// wave sums its whole group, which costs nothing while the other waves of all resident blocks (4 a CU) wait for memory,
// but adds up over rows x group. One launch against a launch for the scores in front, us: kernels of 1536 x 1800 in
// groups of 16 / 1024 rows 23.0 / 24.0 against 23.9 / 28.8; whole advantage computations of 2048 x 2048 in groups of 16 /
// 2048 rows 38.9 / 64.2 against 39.5 / 61.9, of 4096 x 2048 in groups of 16 / 4096 rows 66.0 / 142.8 against
// 63.7 / 110.6, of one group of 8192 x 1800 430 against 274.
bool scores_fit(int64_t n_seqs) { return n_seqs <= 2048; }

// Arguments of adv_gae_kernel from those of areal_advantages_row_stats (with norm: advantages normalised, no row sums).
int adv_gae_args(AdvGaeArgs& a, const float* rewards, int score_mode, float bias, float scaling, float clip,
                        const int64_t* group_offsets, const int64_t* group_rows, int64_t n_groups, int tail_group,
                        int mean_level, int std_level, int unbiased, double eps, const uint8_t* loss_mask,
                        const uint8_t* attn_mask, const float* logp, float* ref_logp, const float* values, int64_t bs,
                        int64_t L, int roll_logp, int estimator, int apply_clamp, int mask_no_eos_with_zero,
                        int ref_in_place, float kl_ctl, float discount, float gae_lambda, float* lm_out, float* old_out,
                        float* kl_out, float* tot_out, int64_t* seqlens_out, uint8_t* no_eos_out, float* advantages,
                        float* returns, double* row_stats, const areal_group_norm_spec* norm) {
  if (bs < 0 || L < 0 || estimator < 1 || estimator > 3 || score_mode < 0 || score_mode > 2) return AREAL_ERR_BAD_ARG;
  if (bs == 0) return AREAL_OK;
  if (L == 0) return AREAL_ERR_BAD_ARG;
  if (!rewards || !loss_mask || !attn_mask || !logp || !lm_out || !old_out || !kl_out || !tot_out || !seqlens_out ||
      !no_eos_out || !advantages || !returns || (!row_stats && norm == nullptr))
    return AREAL_ERR_BAD_ARG;
  if (score_mode == 2 && (!group_offsets || !group_rows || n_groups <= 0)) return AREAL_ERR_BAD_ARG;
  if (score_mode == 2 && (mean_level < 0 || mean_level > 2 || std_level < 0 || std_level > 2)) return AREAL_ERR_BAD_ARG;
  if (score_mode == 2 && (mean_level == LEVEL_BATCH || std_level == LEVEL_BATCH)) return AREAL_ERR_UNSUPPORTED;
  if (!row_sums_fit(bs, L) || (score_mode == 2 && !scores_fit(bs))) return AREAL_ERR_UNSUPPORTED;
  // with the log-probs rolled a thread reads its neighbour's token: not in place
  if (roll_logp && logp == old_out) return AREAL_ERR_BAD_ARG;
  a.p = PrepArgs{loss_mask, attn_mask, logp, ref_logp, rewards, L, roll_logp, estimator, apply_clamp,
                 mask_no_eos_with_zero, ref_in_place, kl_ctl, lm_out, old_out, kl_out, nullptr, nullptr, tot_out,
                 seqlens_out, no_eos_out};
  a.g = GaeArgs{nullptr, values, nullptr, nullptr, nullptr, nullptr, bs * L, (int)bs, L, discount, gae_lambda, advantages,
                returns, 1, row_stats};
  a.score_mode = score_mode;
  a.bias = bias; a.scaling = scaling; a.clip = clip;
  a.score.x = rewards; a.score.n = bs; a.score.goff = group_offsets; a.score.grows = group_rows;
  a.score.G = (int)n_groups; a.score.tail_group = tail_group; a.score.mean_level = mean_level;
  a.score.std_level = std_level; a.score.unbiased = unbiased; a.score.eps = eps;
  if (norm == nullptr) return AREAL_OK;
  if (!norm->group_offsets || norm->n_groups <= 0 || norm->max_group_rows <= 0) return AREAL_ERR_BAD_ARG;
  if (norm->mean_level < 0 || norm->mean_level > 2 || norm->std_level < 0 || norm->std_level > 2) return AREAL_ERR_BAD_ARG;
  if (norm->mean_level == LEVEL_BATCH || norm->std_level == LEVEL_BATCH || norm->leave_one_out || norm->tail_group >= 0 ||
      norm->n_groups > (1 << 30) || norm->max_group_rows > ADV_GROUP_ROWS || L > ADV_NORM_TILES * (int64_t)GAE_TILE)
    return AREAL_ERR_UNSUPPORTED;
  a.norm.goff = norm->group_offsets; a.norm.G = (int)norm->n_groups; a.norm.tail_group = -1;
  a.norm.mean_level = norm->mean_level; a.norm.std_level = norm->std_level; a.norm.unbiased = norm->unbiased;
  a.norm.eps = norm->eps;
  return AREAL_OK;
}
template <bool NORM>
int launch_adv_gae(const AdvGaeArgs& a, hipStream_t stream) {
  const int64_t L = a.p.L;
  const dim3 gr((unsigned)a.g.n_seqs), bl(GAE_THREADS);
  const size_t lds = NORM ? (size_t)ceil_div_i64(L, GAE_TILE) * GAE_TILE * sizeof(float) : 0;
  auto launch = [&](auto one_tile) {
    constexpr bool ONE = decltype(one_tile)::value;
    if (a.p.estimator == 1) hipLaunchKernelGGL((adv_gae_kernel<1, ONE, NORM>), gr, bl, lds, stream, a);
    else if (a.p.estimator == 2) hipLaunchKernelGGL((adv_gae_kernel<2, ONE, NORM>), gr, bl, lds, stream, a);
    else hipLaunchKernelGGL((adv_gae_kernel<3, ONE, NORM>), gr, bl, lds, stream, a);
  };
  if (L <= GAE_TILE) launch(std::true_type{});
  else launch(std::false_type{});
  AREAL_CHECK_LAUNCH();
  return AREAL_OK;
}

}  // namespace

extern "C" {

size_t areal_gae_workspace_bytes(int64_t n_tokens) {
  if (n_tokens <= 0) return 0;
  const int64_t nb = ceil_div_i64(n_tokens, GAE_TILE);
  return (size_t)nb * (sizeof(Map) + 2 * sizeof(double)) + 256;
}

// Generalised advantage estimation over packed sequences.
//   sequences: cu_seqlens [n_seqs+1] (int32), or uniform_len > 0 for a padded [n_seqs, L] array
//   no_eos [n_seqs] (uint8, nullable): bootstrap from the last value of the sequence
//   lambda_seq [n_seqs] (nullable): per-sequence lambda, else the scalar gae_lambda
int areal_gae_packed(const float* rewards, const float* values, const float* loss_mask,
                     const int32_t* cu_seqlens, const uint8_t* no_eos, const float* lambda_seq,
                     int64_t n_tokens, int64_t n_seqs, int64_t uniform_len, float discount,
                     float gae_lambda, float* advantages, float* returns, void* workspace,
                     size_t workspace_bytes, hipStream_t stream) {
  if (n_tokens < 0 || n_seqs < 0) return AREAL_ERR_BAD_ARG;
  if (n_tokens == 0) return AREAL_OK;
  if (!rewards || !values || !loss_mask || !advantages || !returns) return AREAL_ERR_BAD_ARG;
  if (n_seqs == 0 || (uniform_len <= 0 && cu_seqlens == nullptr)) return AREAL_ERR_BAD_ARG;
  if (uniform_len > 0 && uniform_len * n_seqs != n_tokens) return AREAL_ERR_BAD_ARG;
  if (n_seqs > (1 << 30)) return AREAL_ERR_UNSUPPORTED;
  if (workspace == nullptr || workspace_bytes < areal_gae_workspace_bytes(n_tokens))
    return AREAL_ERR_WORKSPACE;
  const int64_t nb = ceil_div_i64(n_tokens, GAE_TILE);
  if (nb > (1 << 30)) return AREAL_ERR_UNSUPPORTED;
  char* wp = (char*)(((uintptr_t)workspace + 255) & ~(uintptr_t)255);
  Map* totals = (Map*)wp;
  double* carry = (double*)(wp + (size_t)nb * sizeof(Map));
  GaeArgs g{rewards, values, loss_mask, cu_seqlens, no_eos, lambda_seq, n_tokens, (int)n_seqs,
            uniform_len, discount, gae_lambda, advantages, returns, 0, nullptr};
  // Measured on 1024 lognormal sequences (1.8 M tokens) / 64 x 16384 / 128 long-tailed up to
  // 32768 / 4 x 32768: tile kernel 19 / 19 / 28 / 24 us, three launches 32 / 21 / 21 / 15 us.
  const int64_t mean_len = n_tokens / n_seqs;
  if (uniform_len <= 0 && mean_len <= 8 * GAE_TILE) {
    // packed sequences: block = tile, the state entering from the right recomputed per tile
    const dim3 grid((unsigned)(ceil_div_i64(nb, 8) * 8));
    if (lambda_seq != nullptr)
      hipLaunchKernelGGL((gae_tile_kernel<true, false>), grid, dim3(GAE_THREADS), 0, stream, g);
    else
      hipLaunchKernelGGL((gae_tile_kernel<false, false>), grid, dim3(GAE_THREADS), 0, stream, g);
    AREAL_CHECK_LAUNCH();
    return AREAL_OK;
  }
  // padded rows: blocks that own whole rows, as long as there are rows enough to fill the chip
  // or the rows are short (a block walks its row's tiles one after the other)
  if (uniform_len > 0 && uniform_len <= 64 * (int64_t)GAE_TILE &&
      (n_seqs >= 256 || uniform_len <= 4 * GAE_TILE)) {
    g.block_per_seq = uniform_len >= GAE_TILE;
    const int64_t grid = g.block_per_seq ? n_seqs : ceil_div_i64(nb, 8) * 8;
    launch_gae_owned<false>(g, grid, stream);
    AREAL_CHECK_LAUNCH();
    return AREAL_OK;
  }
  // long sequences: reduce-then-scan over all tokens
  hipLaunchKernelGGL(gae_block_total_kernel, dim3((unsigned)nb), dim3(GAE_THREADS), 0, stream, g,
                     totals);
  AREAL_CHECK_LAUNCH();
  hipLaunchKernelGGL(gae_carry_kernel, dim3(1), dim3(GAE_THREADS), 0, stream, totals, (int)nb,
                     carry);
  AREAL_CHECK_LAUNCH();
  hipLaunchKernelGGL(gae_apply_kernel, dim3((unsigned)nb), dim3(GAE_THREADS), 0, stream, g, carry);
  AREAL_CHECK_LAUNCH();
  return AREAL_OK;
}

// areal_gae_packed on a padded [n_seqs, uniform_len] batch (values may be null: no critic, all zero), which
// also leaves in row_stats [5][n_seqs] (fp64) the masked sums of each row's
// advantages that areal_group_norm_from_row_stats turns into means and deviations: the
// statistics pass of a normalisation of the advantages under the same mask, at no extra traffic.
int areal_gae_padded_row_stats(const float* rewards, const float* values, const float* loss_mask,
                               const uint8_t* no_eos, const float* lambda_seq, int64_t n_seqs,
                               int64_t uniform_len, float discount, float gae_lambda,
                               float* advantages, float* returns, double* row_stats,
                               hipStream_t stream) {
  if (n_seqs < 0 || uniform_len < 0) return AREAL_ERR_BAD_ARG;
  if (n_seqs == 0 || uniform_len == 0) return AREAL_OK;
  if (!rewards || !loss_mask || !advantages || !returns || !row_stats) return AREAL_ERR_BAD_ARG;
  if (!row_sums_fit(n_seqs, uniform_len)) return AREAL_ERR_UNSUPPORTED;
  GaeArgs g{rewards, values, loss_mask, nullptr, no_eos, lambda_seq, n_seqs * uniform_len, (int)n_seqs,
            uniform_len, discount, gae_lambda, advantages, returns, 1, row_stats};
  launch_gae_owned<true>(g, n_seqs, stream);
  AREAL_CHECK_LAUNCH();
  return AREAL_OK;
}

// Packed GAE that also leaves the statistics pass of a group normalisation of its advantages:
// groups are runs of whole sequences, group_offsets [n_groups + 1] (int64, device) their token
// offsets (group_offsets[0] = 0, group_offsets[n_groups] = n_tokens). segment_stats receives
// [5][slots][4] fp64 sums (slots = 2048-token tiles + groups) for
// areal_group_norm_from_segment_stats. One launch. AREAL_ERR_UNSUPPORTED when the batch is not one
// for the single-pass kernel (sequences longer than 16384 tokens on average) or the groups are
// shorter than 256 tokens on average: the caller then runs areal_gae_packed and areal_group_norm.
size_t areal_gae_segment_stats_bytes(int64_t n_tokens, int64_t n_groups) {
  if (n_tokens <= 0 || n_groups <= 0) return 0;
  return (size_t)5 * GAE_SEG_WAVES * (size_t)(ceil_div_i64(n_tokens, GAE_TILE) + n_groups) * sizeof(double);
}

int areal_gae_packed_group_stats(const float* rewards, const float* values, const float* loss_mask,
                                 const int32_t* cu_seqlens, const uint8_t* no_eos,
                                 const float* lambda_seq, int64_t n_tokens, int64_t n_seqs,
                                 float discount, float gae_lambda, const int64_t* group_offsets,
                                 int64_t n_groups, float* advantages, float* returns,
                                 double* segment_stats, size_t segment_stats_bytes,
                                 hipStream_t stream) {
  if (n_tokens < 0 || n_seqs < 0 || n_groups < 0) return AREAL_ERR_BAD_ARG;
  if (n_tokens == 0) return AREAL_OK;
  if (!rewards || !values || !loss_mask || !advantages || !returns || !cu_seqlens || !group_offsets ||
      !segment_stats || n_seqs == 0 || n_groups == 0)
    return AREAL_ERR_BAD_ARG;
  if (n_seqs > (1 << 30) || n_groups > (1 << 30)) return AREAL_ERR_UNSUPPORTED;
  const int64_t nb = ceil_div_i64(n_tokens, GAE_TILE);
  if (nb > (1 << 30)) return AREAL_ERR_UNSUPPORTED;
  if (n_tokens / n_seqs > 8 * GAE_TILE || n_tokens / n_groups < 256) return AREAL_ERR_UNSUPPORTED;
  if (segment_stats_bytes < areal_gae_segment_stats_bytes(n_tokens, n_groups)) return AREAL_ERR_WORKSPACE;
  GaeArgs g{rewards, values, loss_mask, cu_seqlens, no_eos, lambda_seq, n_tokens, (int)n_seqs,
            0, discount, gae_lambda, advantages, returns, 0, nullptr};
  g.goff = group_offsets; g.n_groups = (int)n_groups; g.seg_stats = segment_stats;
  g.seg_slots = nb + n_groups;
  const dim3 grid((unsigned)(ceil_div_i64(nb, 8) * 8));
  if (lambda_seq != nullptr)
    hipLaunchKernelGGL((gae_tile_kernel<true, true>), grid, dim3(GAE_THREADS), 0, stream, g);
  else
    hipLaunchKernelGGL((gae_tile_kernel<false, true>), grid, dim3(GAE_THREADS), 0, stream, g);
  AREAL_CHECK_LAUNCH();
  return AREAL_OK;
}

// areal_gae_packed_group_stats followed by the group normalisation of its advantages, in two launches that
// need nothing from the host: group j is the sequences [group_first[j], group_first[j + 1]) (int64,
// device; group_first[n_groups] = n_seqs), group_rows their numbers. Levels and unsupported combinations
// as areal_group_norm_from_segment_stats, unsupported batches as areal_gae_packed_group_stats; values may be null.
int areal_gae_packed_normalized(const float* rewards, const float* values, const float* loss_mask,
                                const int32_t* cu_seqlens, const uint8_t* no_eos, const float* lambda_seq,
                                int64_t n_tokens, int64_t n_seqs, float discount, float gae_lambda,
                                const int64_t* group_first, const int64_t* group_rows, int64_t n_groups,
                                int tail_group, int mean_level, int std_level, int unbiased, double eps,
                                float* advantages, float* returns, float* normalized, double* segment_stats,
                                size_t segment_stats_bytes, hipStream_t stream) {
  if (n_tokens < 0 || n_seqs < 0 || n_groups < 0) return AREAL_ERR_BAD_ARG;
  if (n_tokens == 0) return AREAL_OK;
  if (!rewards || !loss_mask || !advantages || !returns || !normalized || !cu_seqlens || !group_first ||
      !group_rows || !segment_stats || n_seqs == 0 || n_groups == 0)
    return AREAL_ERR_BAD_ARG;
  if (mean_level < 0 || mean_level > 2 || std_level < 0 || std_level > 2) return AREAL_ERR_BAD_ARG;
  if (mean_level == LEVEL_GROUP && std_level == LEVEL_BATCH) return AREAL_ERR_UNSUPPORTED;
  if (n_seqs > (1 << 30) || n_groups > (1 << 30)) return AREAL_ERR_UNSUPPORTED;
  const int64_t nb = ceil_div_i64(n_tokens, GAE_TILE);
  if (nb > (1 << 29)) return AREAL_ERR_UNSUPPORTED;
  if (n_tokens / n_seqs > 8 * GAE_TILE || n_tokens / n_groups < 256) return AREAL_ERR_UNSUPPORTED;
  if (segment_stats_bytes < areal_gae_segment_stats_bytes(n_tokens, n_groups)) return AREAL_ERR_WORKSPACE;
  if (((uintptr_t)advantages | (uintptr_t)loss_mask | (uintptr_t)normalized) & 15) return AREAL_ERR_ALIGNMENT;
  GaeArgs g{rewards, values, loss_mask, cu_seqlens, no_eos, lambda_seq, n_tokens, (int)n_seqs,
            0, discount, gae_lambda, advantages, returns, 0, nullptr};
  g.goff = nullptr; g.gseq = group_first; g.n_groups = (int)n_groups; g.seg_stats = segment_stats;
  g.seg_slots = nb + n_groups;
  const dim3 grid((unsigned)(ceil_div_i64(nb, 8) * 8));
  if (lambda_seq != nullptr)
    hipLaunchKernelGGL((gae_tile_kernel<true, true>), grid, dim3(GAE_THREADS), 0, stream, g);
  else
    hipLaunchKernelGGL((gae_tile_kernel<false, true>), grid, dim3(GAE_THREADS), 0, stream, g);
  AREAL_CHECK_LAUNCH();
  NormArgs a{};
  a.x = advantages; a.mask = loss_mask; a.n = n_tokens; a.goff = nullptr; a.grows = group_rows;
  a.G = (int)n_groups; a.tail_group = tail_group;
  a.mean_level = mean_level; a.std_level = std_level; a.unbiased = unbiased; a.eps = eps;
  a.part = segment_stats; a.out = normalized; a.closed_form = 1;
  a.part_tile = GAE_TILE; a.part_slots = g.seg_slots;
  const GroupOffsets go{nullptr, group_first, cu_seqlens, 0};
  hipLaunchKernelGGL(norm_apply_seg_kernel, dim3((unsigned)ceil_div_i64(n_tokens, SEG_APPLY_ELEMS)), dim3(NORM_THREADS),
                     0, stream, a, go);
  AREAL_CHECK_LAUNCH();
  return AREAL_OK;
}

// areal_gae_packed_normalized in one launch where it can be (gae_tile_norm_kernel), else in its two. max_group_seqs: the
// sequences of the largest group; wait_us as areal_group_norm_spec.
size_t areal_gae_packed_normalized_workspace_bytes(int64_t n_tokens, int64_t n_groups) {
  if (n_tokens <= 0 || n_groups <= 0) return 0;
  const size_t tiles = (size_t)ceil_div_i64(n_tokens, GAE_TILE);
  const size_t sums = round_up_i64((int64_t)(tiles + (size_t)n_groups) * (SUMS_PITCH + 2), MAP_PITCH);
  return std::max((sums + tiles * GAE_SEG_WAVES * MAP_PITCH) * sizeof(uint64_t),
                  areal_gae_segment_stats_bytes(n_tokens, n_groups)) + 256;
}
int areal_gae_packed_normalized_ex(const float* rewards, const float* values, const float* loss_mask,
                                   const int32_t* cu_seqlens, const uint8_t* no_eos, const float* lambda_seq,
                                   int64_t n_tokens, int64_t n_seqs, float discount, float gae_lambda,
                                   const int64_t* group_first, const int64_t* group_rows, int64_t n_groups,
                                   int64_t max_group_seqs, int tail_group, int mean_level, int std_level, int unbiased,
                                   double eps, int wait_us, float* advantages, float* returns, float* normalized,
                                   void* workspace, size_t workspace_bytes, hipStream_t stream) {
  if (n_tokens < 0 || n_seqs < 0 || n_groups < 0) return AREAL_ERR_BAD_ARG;
  if (n_tokens == 0) return AREAL_OK;
  if (!rewards || !loss_mask || !advantages || !returns || !normalized || !cu_seqlens || !group_first ||
      !group_rows || n_seqs == 0 || n_groups == 0)
    return AREAL_ERR_BAD_ARG;
  if (workspace == nullptr || workspace_bytes < areal_gae_packed_normalized_workspace_bytes(n_tokens, n_groups))
    return AREAL_ERR_WORKSPACE;
  uint64_t* const ws = (uint64_t*)(((uintptr_t)workspace + 255) & ~(uintptr_t)255);
  const int64_t nb = ceil_div_i64(n_tokens, GAE_TILE);
  hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
  const bool known = hipStreamIsCapturing(stream, &capture) == hipSuccess;
  if (!known) (void)hipGetLastError();
  // While all tiles are on the chip at once (4 blocks a CU) one launch is the better one for groups of any size measured,
  // up to 64 tiles; with more tiles the blocks that wait keep those that they wait for from starting. Two launches / one,
  // us (tiles, tiles a group): 875, 14: 28.2 / 25.1; 875, 55: 28.8 / 27.5; 1024, 16: 31.7 / 26.9; 1024, 64: 32.7 / 28.6; 1040, 4:
  // 38.0 / 33.3; 2000, 4: 56.5 / 52.0; 2000, 8: 55.0 / 53.0, of shorter sequences 49.7 / 50.6; 1200, 16: 40.1 / 39.2; 2000, 16: 54.2 /
  // 58.6; 2000, 32: 53.1 / 64.0; 2048, 64: 54.0 / 115.3. The mean length is bounded as areal_gae_packed's, by what making all maps in each block
  // bears: where they are handed over, longer ones would gain too (whole call of 32 x 32768 in fours 75, in one launch 25).
  const int64_t most_tiles = nb <= GAE_TILES_AT_ONCE ? 64 : 4;
  const bool one = known && capture == hipStreamCaptureStatusNone && tail_group < 0 && mean_level != LEVEL_BATCH &&
                   std_level != LEVEL_BATCH && nb <= (1 << 29) &&
                   max_group_seqs * ceil_div_i64(n_tokens, n_seqs) <= most_tiles * GAE_TILE &&
                   n_tokens / n_seqs <= 8 * GAE_TILE && n_tokens / n_groups >= 256 &&
                   (((uintptr_t)rewards | (uintptr_t)values | (uintptr_t)advantages | (uintptr_t)loss_mask |
                     (uintptr_t)normalized) & 15) == 0;
  if (!one)
    return areal_gae_packed_normalized(rewards, values, loss_mask, cu_seqlens, no_eos, lambda_seq, n_tokens, n_seqs, discount,
                                       gae_lambda, group_first, group_rows, n_groups, tail_group, mean_level, std_level,
                                       unbiased, eps, advantages, returns, normalized, (double*)ws,
                                       areal_gae_segment_stats_bytes(n_tokens, n_groups), stream);
  if (mean_level < 0 || mean_level > 2 || std_level < 0 || std_level > 2) return AREAL_ERR_BAD_ARG;
  GaeNormArgs a{};
  a.g = GaeArgs{rewards, values, loss_mask, cu_seqlens, no_eos, lambda_seq, n_tokens, (int)n_seqs,
                0, discount, gae_lambda, advantages, returns, 0, nullptr};
  a.g.gseq = group_first; a.g.n_groups = (int)n_groups; a.g.seg_slots = nb + n_groups;
  a.norm.grows = group_rows; a.norm.G = (int)n_groups; a.norm.tail_group = -1;
  a.norm.mean_level = mean_level; a.norm.std_level = std_level; a.norm.unbiased = unbiased; a.norm.eps = eps;
  a.norm.out = normalized;
  a.sums = ws;
  a.flags = ws + SUMS_PITCH * a.g.seg_slots;
  a.left = a.flags + a.g.seg_slots;
  a.maps.at = ws + round_up_i64(a.g.seg_slots * (SUMS_PITCH + 2), MAP_PITCH);
  a.call = next_call_number();
  a.maps.call = a.call;
  a.maps.ticks = group_wait_ticks(wait_us);
  a.maps.wait = nb <= GAE_TILES_AT_ONCE;  // (a tile that is not on the chip yet is not waited for)
  const dim3 grid((unsigned)(ceil_div_i64(nb, 8) * 8));
  if (lambda_seq != nullptr) hipLaunchKernelGGL((gae_tile_norm_kernel<true>), grid, dim3(GAE_THREADS), 0, stream, a);
  else hipLaunchKernelGGL((gae_tile_norm_kernel<false>), grid, dim3(GAE_THREADS), 0, stream, a);
  AREAL_CHECK_LAUNCH();
  return AREAL_OK;
}

// Reward scores of a batch: see reward_score_kernel. group_offsets (rows) / group_rows / n_groups as
// areal_group_norm, n_groups 0: no normalisation.
int areal_reward_scores(const float* rewards, int64_t n, float bias, float scaling, float clip,
                        const int64_t* group_offsets, const int64_t* group_rows, int64_t n_groups, int tail_group,
                        int mean_level, int std_level, int unbiased, double eps, float* out, hipStream_t stream) {
  if (n < 0 || n_groups < 0) return AREAL_ERR_BAD_ARG;
  if (n == 0) return AREAL_OK;
  if (!rewards || !out || (n_groups > 0 && (!group_offsets || !group_rows))) return AREAL_ERR_BAD_ARG;
  if (mean_level < 0 || mean_level > 2 || std_level < 0 || std_level > 2) return AREAL_ERR_BAD_ARG;
  if (mean_level == LEVEL_GROUP && std_level == LEVEL_BATCH) return AREAL_ERR_UNSUPPORTED;
  NormArgs a{};
  a.x = rewards; a.n = n; a.goff = group_offsets; a.grows = group_rows; a.G = (int)n_groups; a.tail_group = tail_group;
  a.mean_level = mean_level; a.std_level = std_level; a.unbiased = unbiased; a.eps = eps; a.out = out;
  if (n_groups > 0 && mean_level != LEVEL_BATCH && std_level != LEVEL_BATCH)
    hipLaunchKernelGGL(reward_score_groups_kernel, dim3((unsigned)ceil_div_i64(n_groups + 1, 4)), dim3(256), 0, stream,
                       a, bias, scaling, clip);
  else
    hipLaunchKernelGGL(reward_score_kernel, dim3(1), dim3(SCORE_THREADS), 0, stream, a, bias, scaling, clip,
                       n_groups > 0 ? 1 : 0);
  AREAL_CHECK_LAUNCH();
  return AREAL_OK;
}

size_t areal_turn_gae_workspace_bytes(int64_t bs, int64_t max_seqlen) {
  if (bs <= 0 || max_seqlen <= 0) return 0;
  return (size_t)bs * ((size_t)(max_seqlen + 1) * sizeof(double) + (size_t)max_seqlen * 3 * sizeof(float)) + 256;
}

// Turn-level GAE on padded [bs, max_seqlen] tensors: rewards, values, loss_mask fp32, turn_ids
// int32 (-1 in prompt / tool gaps), no_eos [bs] (nullable), lambda_seq [bs] (nullable, else the
// scalar). status (device int, zeroed by the caller) receives a bit mask of malformed turn ids
// at active tokens: 1 negative, 2 not smaller than max_seqlen, 4 decreasing.
int areal_turn_gae(const float* rewards, const float* values, const float* loss_mask,
                   const int32_t* turn_ids, const uint8_t* no_eos, const float* lambda_seq,
                   int64_t bs, int64_t max_seqlen, float discount, float gae_lambda,
                   float* advantages, float* returns, int* status, void* workspace,
                   size_t workspace_bytes, hipStream_t stream) {
  if (bs > 0 && max_seqlen > 0 && !values) return AREAL_ERR_BAD_ARG;
  return areal_turn_gae_ex(rewards, values, loss_mask, turn_ids, 0, no_eos, lambda_seq, nullptr, bs, max_seqlen,
                           discount, gae_lambda, advantages, returns, status, workspace, workspace_bytes, stream);
}

// ... with values nullable (all zero), roll_ids (the ids of the next-token convention are turn_ids[:, t + 1] and
// -1 at the end) and addend [bs, max_seqlen] (nullable), which is added to the advantages.
int areal_turn_gae_ex(const float* rewards, const float* values, const float* loss_mask, const int32_t* turn_ids,
                      int roll_ids, const uint8_t* no_eos, const float* lambda_seq, const float* addend, int64_t bs,
                      int64_t max_seqlen, float discount, float gae_lambda, float* advantages, float* returns,
                      int* status, void* workspace, size_t workspace_bytes, hipStream_t stream) {
  if (bs < 0 || max_seqlen < 0) return AREAL_ERR_BAD_ARG;
  if (bs == 0 || max_seqlen == 0) return AREAL_OK;
  if (!rewards || !loss_mask || !turn_ids || !advantages || !returns || !status) return AREAL_ERR_BAD_ARG;
  if (bs > (1 << 30) || max_seqlen > (1 << 30)) return AREAL_ERR_UNSUPPORTED;
  if (workspace == nullptr || workspace_bytes < areal_turn_gae_workspace_bytes(bs, max_seqlen))
    return AREAL_ERR_WORKSPACE;
  char* wp = (char*)(((uintptr_t)workspace + 255) & ~(uintptr_t)255);
  TurnArgs a;
  a.rewards = rewards; a.values = values; a.mask = loss_mask; a.turn_ids = turn_ids;
  a.no_eos = no_eos; a.lam_seq = lambda_seq; a.bs = bs; a.L = max_seqlen;
  a.discount = discount; a.lam = gae_lambda; a.adv = advantages; a.ret = returns;
  a.ws_prefix = (double*)wp;
  a.ws_val = (float*)(wp + (size_t)bs * (size_t)(max_seqlen + 1) * sizeof(double));
  a.ws_adv = a.ws_val + (size_t)bs * max_seqlen;
  a.ws_ret = a.ws_adv + (size_t)bs * max_seqlen;
  a.status = status;
  a.roll = roll_ids; a.addend = addend;
  auto launch = [&](auto threads) {
    hipLaunchKernelGGL((turn_gae_kernel<decltype(threads)::value>), dim3((unsigned)bs), dim3(decltype(threads)::value), 0,
                       stream, a);
  };
  // A row in as few tiles as can be while all rows' blocks are resident (rows x slots, us with blocks of 256 / 512 /
  // 1024 threads: 128 x 8192 37.5 / 26.9 / 20.8, 512 x 4096 24.6 / 19.9 / 19.1, 1024 x 2001 18.3 / 16.7 / -; but
  // 1024 x 8192 58.4 / 67.1 / 80.9).
  if (max_seqlen > 512 * TURN_ITEMS && bs <= 512) launch(std::integral_constant<int, 1024>{});
  else if (max_seqlen > 256 * TURN_ITEMS && max_seqlen <= 512 * TURN_ITEMS && bs <= 1024)
    launch(std::integral_constant<int, 512>{});
  else launch(std::integral_constant<int, 256>{});
  AREAL_CHECK_LAUNCH();
  return AREAL_OK;
}

// token_lengths[b] = active tokens of row b; turn_counts[b] = distinct turn ids among them (0
// when turn_ids is null). status as in areal_turn_gae.
int areal_gae_lambda_context(const float* loss_mask, const int32_t* turn_ids, int64_t bs,
                             int64_t max_seqlen, int64_t* token_lengths, int64_t* turn_counts,
                             int* status, hipStream_t stream) {
  if (bs < 0 || max_seqlen < 0) return AREAL_ERR_BAD_ARG;
  if (bs == 0) return AREAL_OK;
  if (!loss_mask || !token_lengths || !turn_counts || !status) return AREAL_ERR_BAD_ARG;
  hipLaunchKernelGGL(gae_context_kernel, dim3((unsigned)bs), dim3(TURN_THREADS), 0, stream,
                     loss_mask, turn_ids, max_seqlen, token_lengths, turn_counts, status);
  AREAL_CHECK_LAUNCH();
  return AREAL_OK;
}

// Blocks per group: 4096 to 8192 elements per block, and at most 2048 partials per array in all
// (every block of the later passes sums them) unless there are more groups than that.
// (5 blocks of these kernels fit a CU at a time: beyond 1280 blocks a second, partly empty round
// starts, so larger inputs take 8192 elements per block.)
static int norm_nsplit(int64_t n_groups, int64_t max_group_len) {
  int64_t s = ceil_div_i64(max_group_len, 4096);
  if (s * n_groups > 1280) s = ceil_div_i64(max_group_len, 8192);
  const int64_t cap = n_groups >= 2048 ? 1 : 2048 / n_groups;
  if (s > cap) s = cap;
  if (s < 1) s = 1;
  return (int)s;
}

size_t areal_group_norm_workspace_bytes(int64_t n_groups, int64_t max_group_len) {
  if (n_groups <= 0) return 0;
  return (size_t)5 * n_groups * norm_nsplit(n_groups, max_group_len) * sizeof(double) + 256;
}

// Normalization(x, mask, groups): levels 0 = none, 1 = batch, 2 = group.
//   group_offsets [G+1] int64 element offsets (device) partitioning [0, n);
//   group_rows [G] int64 (device): number of rows (samples) of each group;
//   tail_group: index of a group made of rows that belong to no group (mean 0, std 0 at group
//   level, still part of batch statistics), or -1.
int areal_group_norm(const float* x, const float* mask, int64_t n, const int64_t* group_offsets,
                     const int64_t* group_rows, int64_t n_groups, int64_t max_group_len,
                     int tail_group, int mean_level, int std_level, int leave_one_out,
                     int unbiased, double eps, float* out, void* workspace,
                     size_t workspace_bytes, hipStream_t stream) {
  if (n < 0 || n_groups < 0) return AREAL_ERR_BAD_ARG;
  if (n == 0) return AREAL_OK;
  if (!x || !out || !group_offsets || !group_rows || n_groups == 0) return AREAL_ERR_BAD_ARG;
  if (mean_level < 0 || mean_level > 2 || std_level < 0 || std_level > 2) return AREAL_ERR_BAD_ARG;
  if (n_groups > 65535 * 16) return AREAL_ERR_UNSUPPORTED;
  if (workspace == nullptr ||
      workspace_bytes < areal_group_norm_workspace_bytes(n_groups, max_group_len))
    return AREAL_ERR_WORKSPACE;
  NormArgs a;
  a.x = x; a.mask = mask; a.n = n; a.goff = group_offsets; a.grows = group_rows;
  a.G = (int)n_groups; a.tail_group = tail_group; a.nsplit = norm_nsplit(n_groups, max_group_len);
  a.mean_level = mean_level; a.std_level = std_level; a.leave1out = leave_one_out;
  a.unbiased = unbiased; a.eps = eps;
  a.part = (double*)(((uintptr_t)workspace + 255) & ~(uintptr_t)255);
  a.out = out;
  // Two launches (one statistics pass) whenever every element of a group sees the same mean and a
  // batch-level deviation does not sit on top of per-group means; otherwise the deviations need
  // a pass of their own.
  a.closed_form = (!leave_one_out && !(mean_level == LEVEL_GROUP && std_level == LEVEL_BATCH)) ? 1 : 0;
  a.part_rows = 0; a.row_len = 0; a.part_tile = 0; a.part_slots = 0;
  const dim3 grid((unsigned)n_groups, (unsigned)a.nsplit);
  if (a.closed_form) {
    hipLaunchKernelGGL(norm_stats5_kernel, grid, dim3(NORM_THREADS), 0, stream, a);
    AREAL_CHECK_LAUNCH();
  } else {
    hipLaunchKernelGGL(norm_stats1_kernel, grid, dim3(NORM_THREADS), 0, stream, a);
    AREAL_CHECK_LAUNCH();
    hipLaunchKernelGGL(norm_stats2_kernel, grid, dim3(NORM_THREADS), 0, stream, a);
    AREAL_CHECK_LAUNCH();
  }
  if (a.closed_form)
    hipLaunchKernelGGL(norm_apply_cf_kernel, grid, dim3(NORM_THREADS), 0, stream, a);
  else
    hipLaunchKernelGGL(norm_apply_kernel, grid, dim3(NORM_THREADS), 0, stream, a);
  AREAL_CHECK_LAUNCH();
  return AREAL_OK;
}

// The apply pass of areal_group_norm alone, on a [n_rows, row_len] array whose per-row sums
// (row_stats [5][n_rows], as areal_gae_padded_row_stats leaves them) are already known: one
// launch. Groups are runs of whole rows (group_offsets in elements, multiples of row_len).
// Only for the level combinations that need no second statistics pass: no leave-one-out, and
// not a group-level mean under a batch-level deviation (AREAL_ERR_UNSUPPORTED otherwise).
int areal_group_norm_from_row_stats(const float* x, const float* mask, int64_t n_rows, int64_t row_len,
                                    const int64_t* group_offsets, const int64_t* group_rows,
                                    int64_t n_groups, int64_t max_group_len, int tail_group,
                                    int mean_level, int std_level, int unbiased, double eps,
                                    const double* row_stats, float* out, hipStream_t stream) {
  if (n_rows < 0 || row_len < 0 || n_groups < 0) return AREAL_ERR_BAD_ARG;
  if (n_rows == 0 || row_len == 0) return AREAL_OK;
  if (!x || !out || !group_offsets || !group_rows || !row_stats || n_groups == 0) return AREAL_ERR_BAD_ARG;
  if (mean_level < 0 || mean_level > 2 || std_level < 0 || std_level > 2) return AREAL_ERR_BAD_ARG;
  if (mean_level == LEVEL_GROUP && std_level == LEVEL_BATCH) return AREAL_ERR_UNSUPPORTED;
  if (n_groups > 65535 * 16) return AREAL_ERR_UNSUPPORTED;
  NormArgs a;
  a.x = x; a.mask = mask; a.n = n_rows * row_len; a.goff = group_offsets; a.grows = group_rows;
  a.G = (int)n_groups; a.tail_group = tail_group; a.nsplit = norm_nsplit(n_groups, max_group_len);
  a.mean_level = mean_level; a.std_level = std_level; a.leave1out = 0;
  a.unbiased = unbiased; a.eps = eps;
  a.part = const_cast<double*>(row_stats);
  a.out = out;
  a.closed_form = 1;
  a.part_rows = n_rows; a.row_len = row_len; a.part_tile = 0; a.part_slots = 0;
  const dim3 grid((unsigned)n_groups, (unsigned)a.nsplit);
  hipLaunchKernelGGL(norm_apply_cf_kernel, grid, dim3(NORM_THREADS), 0, stream, a);
  AREAL_CHECK_LAUNCH();
  return AREAL_OK;
}

// The apply pass of areal_group_norm alone on a packed array whose per-segment sums
// (segment_stats, as areal_gae_packed_group_stats leaves them for the same n and group_offsets)
// are already known: one launch. Same level restrictions as areal_group_norm_from_row_stats.
int areal_group_norm_from_segment_stats(const float* x, const float* mask, int64_t n,
                                        const int64_t* group_offsets, const int64_t* group_rows,
                                        int64_t n_groups, int64_t max_group_len, int tail_group,
                                        int mean_level, int std_level, int unbiased, double eps,
                                        const double* segment_stats, float* out, hipStream_t stream) {
  if (n < 0 || n_groups < 0) return AREAL_ERR_BAD_ARG;
  if (n == 0) return AREAL_OK;
  if (!x || !out || !group_offsets || !group_rows || !segment_stats || n_groups == 0) return AREAL_ERR_BAD_ARG;
  if (mean_level < 0 || mean_level > 2 || std_level < 0 || std_level > 2) return AREAL_ERR_BAD_ARG;
  if (mean_level == LEVEL_GROUP && std_level == LEVEL_BATCH) return AREAL_ERR_UNSUPPORTED;
  if (n_groups > 65535 * 16) return AREAL_ERR_UNSUPPORTED;
  NormArgs a;
  a.x = x; a.mask = mask; a.n = n; a.goff = group_offsets; a.grows = group_rows;
  a.G = (int)n_groups; a.tail_group = tail_group;
  // the partial sums do not depend on the split: one round of 16 elements per thread
  int64_t ns = ceil_div_i64(max_group_len, (int64_t)SEG_APPLY_ELEMS);
  if (ns > 65535) ns = 65535;
  if (ns < 1) ns = 1;
  a.nsplit = (int)ns;
  a.mean_level = mean_level; a.std_level = std_level; a.leave1out = 0;
  a.unbiased = unbiased; a.eps = eps;
  a.part = const_cast<double*>(segment_stats);
  a.out = out;
  a.closed_form = 1;
  a.part_rows = 0; a.row_len = 0;
  a.part_tile = GAE_TILE; a.part_slots = ceil_div_i64(n, GAE_TILE) + n_groups;
  const dim3 grid((unsigned)n_groups, (unsigned)a.nsplit);
  hipLaunchKernelGGL(norm_apply_cf_kernel, grid, dim3(NORM_THREADS), 0, stream, a);
  AREAL_CHECK_LAUNCH();
  return AREAL_OK;
}

size_t areal_masked_norm_workspace_bytes(int64_t n) {
  (void)n;
  return (size_t)3 * 256 * sizeof(double) + 256;
}

int areal_masked_norm(const float* x, const float* mask, int64_t n, int unbiased, double eps,
                      float* out, void* workspace, size_t workspace_bytes, hipStream_t stream) {
  if (n < 0) return AREAL_ERR_BAD_ARG;
  if (n == 0) return AREAL_OK;
  if (!x || !out) return AREAL_ERR_BAD_ARG;
  if (workspace == nullptr || workspace_bytes < areal_masked_norm_workspace_bytes(n))
    return AREAL_ERR_WORKSPACE;
  double* part = (double*)(((uintptr_t)workspace + 255) & ~(uintptr_t)255);
  int64_t nb = ceil_div_i64(n, NORM_THREADS * 8);
  if (nb > 256) nb = 256;
  hipLaunchKernelGGL(masked_norm_stats_kernel, dim3((unsigned)nb), dim3(NORM_THREADS), 0, stream, x,
                     mask, n, part);
  AREAL_CHECK_LAUNCH();
  hipLaunchKernelGGL(masked_norm_apply_kernel, dim3((unsigned)nb), dim3(NORM_THREADS), 0, stream, x,
                     mask, n, (const double*)part, (int)nb, unbiased, eps, out);
  AREAL_CHECK_LAUNCH();
  return AREAL_OK;
}

// masked_normalization over the trailing dimensions: x, mask (nullable), out are [rows, cols].
int areal_masked_norm_rows(const float* x, const float* mask, int64_t rows, int64_t cols,
                           int unbiased, double eps, float* out, hipStream_t stream) {
  if (rows < 0 || cols < 0 || rows > 0x7fffffffLL) return AREAL_ERR_BAD_ARG;
  if (rows == 0 || cols == 0) return AREAL_OK;
  if (!x || !out) return AREAL_ERR_BAD_ARG;
  hipLaunchKernelGGL(masked_norm_rows_kernel, dim3((unsigned)rows), dim3(NORM_THREADS), 0, stream, x,
                     mask, cols, unbiased, eps, out);
  AREAL_CHECK_LAUNCH();
  return AREAL_OK;
}

// Reward shaping in front of GAE on a padded [bs, L] batch; see adv_prep_kernel. loss_mask and
// attn_mask are bytes (nonzero = set); ref_logp, gkl_out and outcome_out may be null. With
// ref_in_place the masked reference log-probs are written back (the reference's `ref_logp *=
// loss_mask`); old_out may be logp itself when roll_logp is 0 (its `old_logp *= loss_mask`).
int areal_advantage_prep(const uint8_t* loss_mask, const uint8_t* attn_mask, const float* logp,
                         float* ref_logp, const float* reward_score, int64_t bs, int64_t L,
                         int roll_logp, int estimator, int apply_clamp, int mask_no_eos_with_zero,
                         int ref_in_place, float kl_ctl, float* lm_out, float* old_out,
                         float* kl_out, float* gkl_out, float* outcome_out, float* tot_out,
                         int64_t* seqlens_out, uint8_t* no_eos_out, hipStream_t stream) {
  if (bs < 0 || L < 0 || bs > 0x7fffffffLL) return AREAL_ERR_BAD_ARG;
  if (estimator < 1 || estimator > 3) return AREAL_ERR_BAD_ARG;
  if (bs == 0) return AREAL_OK;
  if (L == 0) return AREAL_ERR_BAD_ARG;
  if (!loss_mask || !attn_mask || !logp || !reward_score || !lm_out || !old_out || !kl_out ||
      !tot_out || !seqlens_out || !no_eos_out)
    return AREAL_ERR_BAD_ARG;
  PrepArgs a{loss_mask, attn_mask, logp, ref_logp, reward_score, L, roll_logp, estimator,
             apply_clamp, mask_no_eos_with_zero, ref_in_place, kl_ctl, lm_out, old_out, kl_out,
             gkl_out, outcome_out, tot_out, seqlens_out, no_eos_out};
  hipLaunchKernelGGL(adv_prep_kernel, dim3((unsigned)bs), dim3(NORM_THREADS), 0, stream, a);
  AREAL_CHECK_LAUNCH();
  return AREAL_OK;
}

// Reward scores, areal_advantage_prep and areal_gae_padded_row_stats of a padded [bs, L] batch in one launch
// (adv_gae_kernel), with their results. score_mode 0: rewards are the scores; 1: they are shaped first;
// 2: and normalised within groups of rows (group_offsets / group_rows / n_groups / tail_group / levels as
// areal_reward_scores, no level the batch). AREAL_ERR_UNSUPPORTED for the layouts that
// areal_gae_padded_row_stats does not take either (make the three calls) and, in mode 2, for more rows than
// scores_fit (areal_reward_scores first, then mode 0).
int areal_advantages_row_stats(const float* rewards, int score_mode, float bias, float scaling, float clip,
                               const int64_t* group_offsets, const int64_t* group_rows, int64_t n_groups, int tail_group,
                               int mean_level, int std_level, int unbiased, double eps, const uint8_t* loss_mask,
                               const uint8_t* attn_mask, const float* logp, float* ref_logp, const float* values,
                               int64_t bs, int64_t L, int roll_logp, int estimator, int apply_clamp,
                               int mask_no_eos_with_zero, int ref_in_place, float kl_ctl, float discount,
                               float gae_lambda, float* lm_out, float* old_out, float* kl_out, float* tot_out,
                               int64_t* seqlens_out, uint8_t* no_eos_out, float* advantages, float* returns,
                               double* row_stats, hipStream_t stream) {
  AdvGaeArgs a{};
  const int rc = adv_gae_args(a, rewards, score_mode, bias, scaling, clip, group_offsets, group_rows, n_groups, tail_group,
                              mean_level, std_level, unbiased, eps, loss_mask, attn_mask, logp, ref_logp, values, bs, L,
                              roll_logp, estimator, apply_clamp, mask_no_eos_with_zero, ref_in_place, kl_ctl, discount,
                              gae_lambda, lm_out, old_out, kl_out, tot_out, seqlens_out, no_eos_out, advantages, returns,
                              row_stats, nullptr);
  return rc != AREAL_OK || bs == 0 ? rc : launch_adv_gae<false>(a, stream);
}

// areal_advantages_row_stats with the advantages normalised within groups of rows in the same launch (see
// adv_normalise_row; the same bits as areal_group_norm_from_row_stats on its sums). AREAL_ERR_UNSUPPORTED, besides
// what areal_advantages_row_stats does not take: a level of the batch, leave one out, ungrouped rows, groups of more than
// 64 rows, rows of more than 8192 slots, and a stream that is being captured (a graph's replays would all carry one
// call's number, and find the sums of the replay before them).
size_t areal_advantages_normalized_workspace_bytes(int64_t bs) { return bs > 0 ? (size_t)bs * 6 * sizeof(uint64_t) + 256 : 0; }

int areal_advantages_normalized(const float* rewards, int score_mode, float bias, float scaling, float clip,
                                const int64_t* group_offsets, const int64_t* group_rows, int64_t n_groups, int tail_group,
                                int mean_level, int std_level, int unbiased, double eps, const uint8_t* loss_mask,
                                const uint8_t* attn_mask, const float* logp, float* ref_logp, const float* values,
                                int64_t bs, int64_t L, int roll_logp, int estimator, int apply_clamp,
                                int mask_no_eos_with_zero, int ref_in_place, float kl_ctl, float discount,
                                float gae_lambda, float* lm_out, float* old_out, float* kl_out, float* tot_out,
                                int64_t* seqlens_out, uint8_t* no_eos_out, float* advantages, float* returns,
                                const areal_group_norm_spec* norm, void* workspace, size_t workspace_bytes,
                                hipStream_t stream) {
  if (norm == nullptr) return AREAL_ERR_BAD_ARG;
  AdvGaeArgs a{};
  const int rc = adv_gae_args(a, rewards, score_mode, bias, scaling, clip, group_offsets, group_rows, n_groups, tail_group,
                              mean_level, std_level, unbiased, eps, loss_mask, attn_mask, logp, ref_logp, values, bs, L,
                              roll_logp, estimator, apply_clamp, mask_no_eos_with_zero, ref_in_place, kl_ctl, discount,
                              gae_lambda, lm_out, old_out, kl_out, tot_out, seqlens_out, no_eos_out, advantages, returns,
                              nullptr, norm);
  if (rc != AREAL_OK || bs == 0) return rc;
  if (workspace == nullptr || workspace_bytes < areal_advantages_normalized_workspace_bytes(bs)) return AREAL_ERR_WORKSPACE;
  hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(stream, &capture) != hipSuccess) {
    (void)hipGetLastError();
    return AREAL_ERR_UNSUPPORTED;
  }
  if (capture != hipStreamCaptureStatusNone) return AREAL_ERR_UNSUPPORTED;
  a.sums = (uint64_t*)(((uintptr_t)workspace + 255) & ~(uintptr_t)255);
  a.flags = a.sums + 4 * bs;
  a.left = a.flags + bs;
  a.call = next_call_number();
  a.wait_ticks = group_wait_ticks(norm->wait_us);
  return launch_adv_gae<true>(a, stream);
}

}  // extern "C"
