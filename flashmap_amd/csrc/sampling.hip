// The draft step's token selection and noise:
//   - argmax over the vocabulary per row, the first index among equals
//     (flashmap/vllm/fold.py:117-128, split_argmax);
//   - the fused sampler: per row the argmax of its logits (greedy rows) or of
//     logit / T - log(-log u) (Gumbel-max, a sample of softmax(logits / T)) with u from
//     Philox at offset row * V + col (flashmap/sglang/kernels.py:195-247, sample_rows);
//   - keyed standard normals, row i keyed by seeds[rows[i]] * 1000003 + positions[i]
//     (flashmap/vllm/kernels.py:367-410, seeded_normal).
//
// The random stream is Triton's tl.rand / tl.randn, word for word: Philox-4x32 with 10
// rounds (Salmon et al., SC 2011) keyed by the seed's low and high words, counter
// (offset, 0, 0, 0) for the int32 offsets both kernels use; a word x maps to
// (x as int32, negatives folded by ~x) * 4.6566127342e-10f; a normal is
// sqrt(-2 log(max(u1, 1e-7))) * cos(6.2831855f * u2) of the first two words.
//
// Selection, argmax: one 256-thread workgroup per (tile of logits, row) streams the tile
// with 16-byte loads, keys it in registers and reduces (key, index) over the wavefront and
// then the workgroup; a one-wavefront-per-row pass merges the tiles. The sampler: one
// workgroup per (part of a row, row), which draws the noise only where it can matter
// (sample_parts_kernel, sample_plan); the same pass merges the parts. NaN counts as the largest key,
// the first NaN winning (torch.argmax's rule).
#include <math.h>
#include <stdint.h>

#include "fm_device.h"
#include "fm_host.h"

namespace fm {

constexpr int SEL_THREADS = 256;
// Logits per workgroup of the argmax. It is HBM-bound: 64 per thread keep more bytes in
// flight per wavefront (1024 x 151936 bf16 logits in 64 us against 71 us with 32 per thread).
constexpr int SEL_TILE = 16384;
constexpr int NOISE_COLS = 1024;  // columns per workgroup of seeded normals (4 per thread)

enum LogitType { LOGITS_BF16 = 0, LOGITS_F16 = 1, LOGITS_F32 = 2 };

__device__ __forceinline__ void philox4x32_10(uint32_t (&c)[4], uint32_t k0, uint32_t k1) {
#pragma unroll
  for (int r = 0; r < 10; ++r) {
    const uint64_t p0 = (uint64_t)0xD2511F53u * c[0];
    const uint64_t p1 = (uint64_t)0xCD9E8D57u * c[2];
    const uint32_t n0 = (uint32_t)(p1 >> 32) ^ c[1] ^ k0;
    const uint32_t n2 = (uint32_t)(p0 >> 32) ^ c[3] ^ k1;
    c[0] = n0;
    c[1] = (uint32_t)p1;
    c[2] = n2;
    c[3] = (uint32_t)p0;
    k0 += 0x9E3779B9u;
    k1 += 0xBB67AE85u;
  }
}

__device__ __forceinline__ float word_to_uniform(uint32_t w) {
  const int32_t i = (int32_t)w;
  return (float)(i < 0 ? ~i : i) * 4.6566127342e-10f;
}

// (key, index) order: NaN above everything (the first NaN wins), else larger key, then
// smaller index.
__device__ __forceinline__ bool better(float k, int32_t i, float bk, int32_t bi) {
  if (k != k) return bk == bk || i < bi;
  if (bk != bk) return false;
  return k > bk || (k == bk && i < bi);
}

__device__ __forceinline__ void wave_best(float &bk, int32_t &bi) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const float k2 = __shfl_xor(bk, o);
    const int32_t i2 = __shfl_xor(bi, o);
    if (better(k2, i2, bk, bi)) bk = k2, bi = i2;
  }
}

template <int TY>
__device__ __forceinline__ float logit_at(const char *row, int64_t col) {
  if (TY == LOGITS_BF16) return bf16_to_f32(reinterpret_cast<const uint16_t *>(row)[col]);
  if (TY == LOGITS_F16) return (float)reinterpret_cast<const _Float16 *>(row)[col];
  return reinterpret_cast<const float *>(row)[col];
}

// Eight consecutive logits starting at col (16-byte aligned for 2-byte types, two
// 16-byte loads for float32).
template <int TY>
__device__ __forceinline__ void logits8(const char *row, int64_t col, float (&x)[8]) {
  if (TY == LOGITS_F32) {
    const u32x4_t a = load16(row + col * 4), b = load16(row + col * 4 + 16);
#pragma unroll
    for (int j = 0; j < 4; ++j) x[j] = __uint_as_float(a[j]), x[4 + j] = __uint_as_float(b[j]);
  } else {
    const u32x4_t a = load16(row + col * 2);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if (TY == LOGITS_BF16) {
        x[2 * j] = bf16_lo(a[j]);
        x[2 * j + 1] = __uint_as_float(a[j] & 0xFFFF0000u);
      } else {
        // through the by-value helpers: a bit cast applied to the vector element a[j]
        // itself is lowered as a cast of a[0]
        x[2 * j] = f16_lo(a[j]);
        x[2 * j + 1] = f16_hi(a[j]);
      }
    }
  }
}

struct SelectArgs {
  const char *logits;
  int64_t row_bytes;  // row stride in bytes
  int64_t vocab;
  int32_t n_tiles, vec;  // vec: rows 16-byte aligned, 8-logit chunks may be loaded whole
  const float *temps;    // sampling only
  const uint8_t *greedy;
  const int64_t *seed;
  float *best;     // (rows, n_tiles)
  int32_t *index;  // (rows, n_tiles)
};

// A thread's best so far over logits that it visits in increasing index order: a strictly
// larger key, the first one, or a first NaN over a number takes the place (branch-free);
// the full order settles ties between threads.
__device__ __forceinline__ void visit_next(float &bk, int32_t &bi, float key, int32_t col) {
  const bool take = key > bk || bi == INT32_MAX || (key != key && bk == bk);
  bk = take ? key : bk;
  bi = take ? col : bi;
}

// The workgroup's best from each thread's, to slot `slot` of the row.
template <int THREADS>
__device__ __forceinline__ void store_best(const SelectArgs &a, int64_t row, int slot, float bk, int32_t bi) {
  wave_best(bk, bi);
  __shared__ float sk[THREADS / 64];
  __shared__ int32_t si[THREADS / 64];
  const int w = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) sk[w] = bk, si[w] = bi;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int v = 1; v < THREADS / 64; ++v)
      if (better(sk[v], si[v], bk, bi)) bk = sk[v], bi = si[v];
    a.best[row * a.n_tiles + slot] = bk;
    a.index[row * a.n_tiles + slot] = bi;
  }
}

// Per (tile, row): the tile's largest logit and its first index.
template <int TY>
__global__ __launch_bounds__(SEL_THREADS) void select_tiles_kernel(const SelectArgs a) {
  const int tile = blockIdx.x;
  const int64_t row = blockIdx.y;
  const char *src = a.logits + row * a.row_bytes;
  float bk = -INFINITY;
  int32_t bi = INT32_MAX;
  auto visit = [&](int64_t col, float key) { visit_next(bk, bi, key, (int32_t)col); };
  const int64_t base = (int64_t)tile * SEL_TILE;
  constexpr int IT = SEL_TILE / (8 * SEL_THREADS);
  if (a.vec && base + SEL_TILE <= a.vocab) {  // a whole tile: every load in flight first
    float x[IT][8];
#pragma unroll
    for (int it = 0; it < IT; ++it) logits8<TY>(src, base + 8 * ((int64_t)it * SEL_THREADS + threadIdx.x), x[it]);
#pragma unroll
    for (int it = 0; it < IT; ++it)
#pragma unroll
      for (int j = 0; j < 8; ++j) visit(base + 8 * ((int64_t)it * SEL_THREADS + threadIdx.x) + j, x[it][j]);
  } else {  // the vocabulary's last, partial tile (or unaligned rows)
#pragma unroll
    for (int it = 0; it < IT; ++it) {
      const int64_t col0 = base + 8 * ((int64_t)it * SEL_THREADS + threadIdx.x);
      if (col0 >= a.vocab) break;
      if (a.vec && col0 + 8 <= a.vocab) {
        float x[8];
        logits8<TY>(src, col0, x);
#pragma unroll
        for (int j = 0; j < 8; ++j) visit(col0 + j, x[j]);
      } else {
        for (int j = 0; j < 8 && col0 + j < a.vocab; ++j) visit(col0 + j, logit_at<TY>(src, col0 + j));
      }
    }
  }
  store_best<SEL_THREADS>(a, row, tile, bk, bi);
}

// The sampler over part blockIdx.x of row blockIdx.y: every gridDim.x-th tile from there.
//
// A sampled row's key is logit / T plus Gumbel noise of at most 16.64 (u is at most
// 1 - 2^-24), and the noise is what costs: 10 rounds of Philox, two logarithms and an IEEE
// division per logit, against 2 bytes of HBM traffic. So the noise is drawn only for
// logits that can still win: those within 16.64 T of the largest key that any thread of the
// workgroup has seen (an LDS maximum that only rises; a late read of it only costs work). A
// wavefront first draws for its 64 lanes' largest logits of the tile, which sets the
// bound near the tile's best at once, then for the rest that pass it, gathered from the
// lanes into an LDS queue and taken 64 at a time; where most of a single tile pass (flat
// logits), each lane takes its own instead, read again from the caches. The uniform word alone rules most
// of these out before the logarithms. Keys, and so tokens, are those of every logit's own
// noise: what is skipped is below the maximum by more than the bound's rounding. The bound
// is no bound (-inf: nothing is skipped) for temperatures whose product with it could over-
// or underflow. Greedy rows look for the largest logit under the same kind of bound.
//
// How much is left depends on the logits and T: of 151936 normal logits with 24 likely ones
// 1 % to 30 % for T from 0.6 to 1.2. Measured on 1024 x 151936 bf16, us (every logit drawn for
// / this kernel): half the rows greedy, T of 0.6 to 1.2: 209 / 111; all sampled at 0.6 330 /
// 69, 1.2 330 / 189; normal logits of sigma 1 327 / 306, equal logits 328 / 314; all greedy
// 74 / 54. Rows that are not 16-byte aligned are read in whole granules all the same (RowView):
// 1024 x 99999 half greedy 181 (logit by logit) / 82, all greedy 121 / 42.
constexpr float GUMBEL_MAX = 16.64f;
constexpr int SAMPLE_IT = 4;  // 8-logit chunks per thread of a tile
constexpr int sample_tile(int threads) { return 8 * SAMPLE_IT * threads; }
// More than this many of a wavefront's first 512 logits above the bound: past the queue (for
// workgroups of one tile; over several the queue has more to gather and the choice costs more
// than it gives: 1024 x 151936, T = 1.2, 1024 threads 189 us, 208 with it). 1024 x 151936 in
// single tiles, T = 1.2: 267 us at 256, 250 at 400, 252 without; equal logits 318, 318, 338.
constexpr int SAMPLE_DIRECT = 400;
constexpr int SAMPLE_QUEUE = 64 + 4 * 64;  // what a drain leaves and four logits of 64 lanes

struct Pending {
  uint32_t col;
  float x;
};

// Orders a wavefront's own LDS accesses across its lanes (LDS serves a wavefront in order;
// this keeps the compiler from moving them).
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// Floats as integers of the same order (no NaN among them).
__device__ __forceinline__ int32_t ordered(float f) {
  const int32_t i = __float_as_int(f);
  return i ^ ((i >> 31) & 0x7fffffff);
}
__device__ __forceinline__ float unordered(int32_t i) { return __int_as_float(i ^ ((i >> 31) & 0x7fffffff)); }

// Eight consecutive logits as they are stored (few registers while a tile is in flight).
template <int TY>
struct Chunk {
  static constexpr int WORDS = TY == LOGITS_F32 ? 8 : 4, PER_WORD = 8 / WORDS;
  uint32_t w[WORDS];
  // The compiler takes the words as new from here on: the logits decoded before are not
  // kept for a later pass over them (32 registers, which would spill).
  __device__ __forceinline__ void forget() {
#pragma unroll
    for (int q = 0; q < WORDS; ++q) asm volatile("" : "+v"(w[q]));
  }
  __device__ __forceinline__ float at(int j) const {
    const uint32_t v = w[j / PER_WORD];
    if (TY == LOGITS_F32) return __uint_as_float(v);
    if (TY == LOGITS_BF16) return j & 1 ? bf16_hi(v) : bf16_lo(v);
    return j & 1 ? f16_hi(v) : f16_lo(v);
  }
  // -inf in the place of logit j.
  __device__ __forceinline__ void drop(int j) {
    uint32_t &v = w[j / PER_WORD];
    if (TY == LOGITS_F32)
      v = 0xFF800000u;
    else
      v = j & 1 ? (v & 0xFFFFu) | (TY == LOGITS_BF16 ? 0xFF800000u : 0xFC000000u)
                : (v & 0xFFFF0000u) | (TY == LOGITS_BF16 ? 0xFF80u : 0xFC00u);
  }
};

// A row as 16-byte granules from the one its first logit lies in: `skip` logits of that
// granule come before the row, and the last granule may end past it. Loads are of whole
// granules with a logit of the row in them (no allocation ends inside one); the logits
// around the row are dropped after the load.
template <int TY>
struct RowView {
  static constexpr int ES = TY == LOGITS_F32 ? 4 : 2;
  const char *from;
  uint32_t skip, vocab, last;  // last: the row's last granule
  __device__ __forceinline__ RowView(const SelectArgs &a, int64_t row) {
    const char *src = a.logits + row * a.row_bytes;
    skip = (uint32_t)((uintptr_t)src & 15) / ES;
    from = src - skip * ES;
    vocab = (uint32_t)a.vocab;
    last = (uint32_t)(((uint64_t)skip + vocab - 1) * ES / 16);
  }
  // Chunk g: the logits of columns 8 g - skip to 8 g - skip + 7.
  __device__ __forceinline__ Chunk<TY> chunk(uint32_t g) const {
    Chunk<TY> c;
#pragma unroll
    for (int h = 0; h < ES / 2; ++h) {
      const uint32_t n = g * (ES / 2) + h;
      const u32x4_t v = load16(from + 16 * (uint64_t)(n < last ? n : last));
#pragma unroll
      for (int q = 0; q < 4; ++q) c.w[4 * h + q] = v[q];
    }
    return c;
  }
  // Whether some of n chunks from g on reach past either end.
  __device__ __forceinline__ bool edge(uint32_t g, uint32_t n) const {
    return (g == 0 && skip != 0) || 8 * ((uint64_t)g + n) > (uint64_t)skip + vocab;
  }
  __device__ __forceinline__ void trim(Chunk<TY> &c, uint32_t g) const {
#pragma unroll
    for (int j = 0; j < 8; ++j)
      if (8 * g - skip + j >= vocab) c.drop(j);
  }
};

// The largest of a thread's logits of a tile (NaN aside) and whether one is NaN.
template <int TY>
__device__ __forceinline__ float tile_max(Chunk<TY> (&x)[SAMPLE_IT], bool &nan) {
  float m = -INFINITY;
  nan = false;
#pragma unroll
  for (int it = 0; it < SAMPLE_IT; ++it) {
#pragma unroll
    for (int j = 0; j < 8; j += 2) {
      const float p = x[it].at(j), q = x[it].at(j + 1);
      m = fmaxf(m, fmaxf(p, q));
      nan |= __builtin_isunordered(p, q);
    }
    x[it].forget();
  }
  return m;
}

__device__ __forceinline__ float sample_uniform(uint32_t offset, uint64_t seed) {
  uint32_t c[4] = {offset, 0u, 0u, 0u};
  philox4x32_10(c, (uint32_t)seed, (uint32_t)(seed >> 32));
  return word_to_uniform(c[0]);
}
__device__ __forceinline__ float sample_key(float x, float temp, float u) { return x / temp - logf(-logf(u)); }

// A row of at most a chunk per thread.
template <int TY, int THREADS>
__device__ __forceinline__ void sample_short(const SelectArgs &a, const RowView<TY> &view, int64_t row) {
  const Chunk<TY> c = view.chunk(threadIdx.x);
  const bool noisy = a.greedy[row] == 0;
  const float temp = a.temps[row];
  const uint64_t seed = (uint64_t)a.seed[0];
  const uint32_t row_off = (uint32_t)row * view.vocab, col0 = 8 * threadIdx.x - view.skip;
  float bk = -INFINITY;
  int32_t bi = INT32_MAX;
  if (8 * threadIdx.x < view.skip + view.vocab) {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      float key = c.at(j);
      if (noisy) key = sample_key(key, temp, sample_uniform(row_off + col0 + j, seed));
      if (col0 + j < view.vocab) visit_next(bk, bi, key, (int32_t)(col0 + j));
    }
  }
  store_best<THREADS>(a, row, blockIdx.x, bk, bi);
}

// SEVERAL: tiles per workgroup; else one.
template <int TY, int THREADS, bool SEVERAL>
__global__ __launch_bounds__(THREADS, TY == LOGITS_F32 ? 4 : 8) void sample_parts_kernel(const SelectArgs a) {
  constexpr uint32_t CHUNKS = SAMPLE_IT * THREADS;  // of a tile
  constexpr uint32_t STEP = 8 * THREADS;            // columns between a thread's chunks
  __shared__ Pending queues[THREADS / 64][SAMPLE_QUEUE];
  __shared__ int32_t bound;
  const int64_t row = blockIdx.y;
  const RowView<TY> view(a, row);
  const uint32_t chunks = (view.skip + view.vocab + 7) / 8, hop = gridDim.x * CHUNKS;
  if (!SEVERAL && chunks <= THREADS) {  // a chunk per thread: every logit drawn for, no bound
    sample_short<TY, THREADS>(a, view, row);
    return;
  }
  // This thread's logits of the tile of chunks from g on: columns col0_of(g) + it * STEP + j.
  auto load = [&](Chunk<TY>(&x)[SAMPLE_IT], uint32_t g) {
#pragma unroll
    for (int it = 0; it < SAMPLE_IT; ++it) x[it] = view.chunk(g + it * THREADS + threadIdx.x);
  };
  auto trim = [&](Chunk<TY>(&x)[SAMPLE_IT], uint32_t g) {
    if (!view.edge(g, CHUNKS)) return;
#pragma unroll
    for (int it = 0; it < SAMPLE_IT; ++it) view.trim(x[it], g + it * THREADS + threadIdx.x);
  };
  auto col0_of = [&](uint32_t g) { return 8 * (g + (uint32_t)threadIdx.x) - view.skip; };
  // The first tile is on its way before the row's own values are looked at.
  const uint32_t first = blockIdx.x * CHUNKS;
  Chunk<TY> x[SAMPLE_IT];
  load(x, first);
  const bool noisy = a.greedy[row] == 0;
  const float temp = a.temps[row];
  const uint64_t seed = (uint64_t)a.seed[0];
  if (threadIdx.x == 0) bound = ordered(-INFINITY);
  if (SEVERAL || noisy) __syncthreads();
  trim(x, first);
  float bk = -INFINITY;
  int32_t bi = INT32_MAX;
  const int lane = threadIdx.x & 63;
  auto raise = [&](float key) {  // the bound takes this wavefront's largest key (NaN aside)
    key = key == key ? key : -INFINITY;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) key = fmaxf(key, __shfl_xor(key, o));
    if (lane == 0) atomicMax(&bound, ordered(key));
    wave_lds_fence();
  };
  auto bound_now = [&] { return unordered(*(volatile __attribute__((address_space(3))) int32_t *)&bound); };
  if (!noisy) {  // the largest logit: tiles without one that reaches the bound are passed over
    Chunk<TY> next[SAMPLE_IT];  // SEVERAL: the next tile in flight
    for (uint32_t g = first;;) {
      if (SEVERAL && g + hop < chunks) load(next, g + hop);
      bool nan;
      const float m = tile_max<TY>(x, nan);
      if (!SEVERAL || g == first || __ballot(!(m < bound_now()) || nan) != 0) {
        const uint32_t col0 = col0_of(g);
        if (__ballot(nan || m == -INFINITY) == 0) {
          uint32_t at = 0;
#pragma unroll
          for (int it = SAMPLE_IT - 1; it >= 0; --it)
#pragma unroll
            for (int j = 7; j >= 0; --j) at = x[it].at(j) == m ? it * STEP + j : at;
          visit_next(bk, bi, m, (int32_t)(col0 + at));
        } else {
#pragma unroll
          for (int it = 0; it < SAMPLE_IT; ++it)
#pragma unroll
            for (int j = 0; j < 8; ++j)
              if (col0 + it * STEP + j < view.vocab) visit_next(bk, bi, x[it].at(j), (int32_t)(col0 + it * STEP + j));
        }
        if (SEVERAL && g + hop < chunks) raise(bk);
      }
      g += hop;
      if (!SEVERAL || g >= chunks) break;
#pragma unroll
      for (int it = 0; it < SAMPLE_IT; ++it) x[it] = next[it];
      trim(x, g);
    }
    store_best<THREADS>(a, row, blockIdx.x, bk, bi);
    return;
  }
  // int32 offsets row * V + col, as the reference's kernel forms them
  const uint32_t row_off = (uint32_t)row * view.vocab;
  Pending *queue = queues[wave_id()];
  int queued = 0;  // wave-uniform
  const bool boundable = temp > 1e-30f && temp < 1e30f;
  const float inv_temp = 1.f / temp;
  float low = -INFINITY;   // logits below it cannot win
  float need = -INFINITY;  // the bound less its slack (see visit)
  auto uniform = [&](uint32_t col) { return sample_uniform(row_off + col, seed); };
  auto keyed = [&](float x, float u) { return sample_key(x, temp, u); };
  // Visits come in any order here: the full order of keys and indices. A key of at least b
  // has -log(u) <= exp(x / T - b), and 1 - u <= -log(u): past exp of the slack above it (2 %,
  // and 2e-6 of b for the roundings), the word alone rules the logit out.
  auto loses = [&](float x, float u) {
    return 1.f - u > __builtin_amdgcn_exp2f((x * inv_temp - need) * 1.44269504f);
  };
  auto visit = [&](uint32_t col, float x, float u) {
    const float key = keyed(x, u);
    if (col < view.vocab && better(key, (int32_t)col, bk, bi)) bk = key, bi = (int32_t)col;
  };
  auto lower = [&] {
    const float b = bound_now();
    const float at = (b - GUMBEL_MAX) * temp;
    // 1e-6 of it: the roundings of the quotient, of the key and of this product
    low = boundable ? at - fabsf(at) * 1e-6f : -INFINITY;
    if (low != low) low = -INFINITY;
    need = boundable ? b - (fabsf(b) + GUMBEL_MAX) * 2e-6f - 0.02f : -INFINITY;
    if (need != need) need = -INFINITY;
  };
  auto drain = [&](int keep) {
    wave_lds_fence();
    while (queued > keep) {
      const int n = queued < 64 ? queued : 64;
      queued -= n;
      if (lane < n) {
        const Pending p = queue[queued + lane];
        const float u = uniform(p.col);
        if (!loses(p.x, u)) visit(p.col, p.x, u);
      }
    }
    wave_lds_fence();
  };
  for (uint32_t g = first;;) {
    const uint32_t col0 = col0_of(g);
    bool take = true;
    if (SEVERAL && g != first) {
      lower();
      bool any = false;
#pragma unroll
      for (int it = 0; it < SAMPLE_IT; ++it) {
#pragma unroll
        for (int j = 0; j < 8; ++j) any |= !(x[it].at(j) < low);
        x[it].forget();
      }
      take = __ballot(any) != 0;
    }
    if (take) {
      float top = x[0].at(0);
      uint32_t at = 0;
#pragma unroll
      for (int it = 0; it < SAMPLE_IT; ++it) {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const bool more = x[it].at(j) > top;
          top = more ? x[it].at(j) : top;
          at = more ? it * STEP + j : at;
        }
        x[it].forget();
      }
      raise(keyed(top, uniform(col0 + at)));  // around the row top is -inf: no bound from it
      if (g == first) __syncthreads();        // every wavefront's, before any logit is taken
      lower();
      int likely = 0;  // of 512 logits
      if constexpr (!SEVERAL) {
#pragma unroll
        for (int j = 0; j < 8; ++j) likely += __popcll(__ballot(!(x[0].at(j) < low)));
        x[0].forget();
      }
      if (!SEVERAL && likely > SAMPLE_DIRECT) {  // most can win: each lane takes its own, without the queue
#pragma unroll 1
        for (uint32_t h = g; h < g + CHUNKS && h < chunks; h += THREADS) {
          if (h + threadIdx.x < chunks) {
            Chunk<TY> c = view.chunk(h + threadIdx.x);
            if (view.edge(h, THREADS)) view.trim(c, h + threadIdx.x);
#pragma unroll
            for (int j = 0; j < 8; j += 4) {  // four at a time: their Philox rounds overlap
              float u[4];
              bool any = false;
#pragma unroll
              for (int k = 0; k < 4; ++k) {
                u[k] = uniform(col0_of(h) + j + k);
                any |= !loses(c.at(j + k), u[k]);
              }
              if (any) {
#pragma unroll
                for (int k = 0; k < 4; ++k)
                  if (!loses(c.at(j + k), u[k])) visit(col0_of(h) + j + k, c.at(j + k), u[k]);
              }
            }
          }
          if (h + THREADS < chunks) {
            raise(bk);
            lower();
          }
        }
      } else {
#pragma unroll
        for (int it = 0; it < SAMPLE_IT; ++it) {
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            const bool can = !(x[it].at(j) < low);
            const uint64_t mask = __ballot(can);
            if (mask != 0) {
              const int before =
                  __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0));
              if (can) queue[queued + before] = Pending{col0 + it * STEP + j, x[it].at(j)};
              queued += __popcll(mask);
            }
            if ((j & 3) == 3 && queued >= 64) drain(63);
          }
        }
      }
    }
    g += hop;
    if (!SEVERAL || g >= chunks) break;
    load(x, g);
    trim(x, g);
  }
  drain(0);
  store_best<THREADS>(a, row, blockIdx.x, bk, bi);
}

// Per row (one wavefront): the best of its tiles.
__global__ __launch_bounds__(64) void select_rows_kernel(const float *best, const int32_t *index, int32_t n_tiles,
                                                         int64_t *out) {
  const int64_t row = blockIdx.x;
  float bk = -INFINITY;
  int32_t bi = INT32_MAX;
  for (int t = threadIdx.x; t < n_tiles; t += 64) {
    const float k = best[row * n_tiles + t];
    const int32_t i = index[row * n_tiles + t];
    if (better(k, i, bk, bi)) bk = k, bi = i;
  }
  wave_best(bk, bi);
  if (threadIdx.x == 0) out[row] = bi;
}

struct NoiseArgs {
  const int64_t *seeds;
  const void *rows;
  const void *positions;
  int32_t rows_64, pos_64;  // index widths: int64 (1) or int32 (0)
  int64_t n_cols, out_stride;
  float scale;
  float *out;
};

__global__ __launch_bounds__(256) void seeded_normal_kernel(const NoiseArgs a) {
  const int64_t row = blockIdx.y;
  const int64_t state = a.rows_64 ? reinterpret_cast<const int64_t *>(a.rows)[row]
                                  : (int64_t)reinterpret_cast<const int32_t *>(a.rows)[row];
  const int64_t pos = a.pos_64 ? reinterpret_cast<const int64_t *>(a.positions)[row]
                               : (int64_t)reinterpret_cast<const int32_t *>(a.positions)[row];
  const uint64_t seed = state >= 0 ? (uint64_t)a.seeds[state] : 0ull;
  const uint64_t key = seed * 1000003ull + (uint64_t)pos;  // int64 arithmetic, wrapping
  const uint32_t k0 = (uint32_t)key, k1 = (uint32_t)(key >> 32);
  float *dst = a.out + row * a.out_stride;
#pragma unroll
  for (int k = 0; k < NOISE_COLS / 256; ++k) {
    const int64_t col = (int64_t)blockIdx.x * NOISE_COLS + k * 256 + threadIdx.x;
    if (col >= a.n_cols) break;
    uint32_t c[4] = {(uint32_t)col, 0u, 0u, 0u};
    philox4x32_10(c, k0, k1);
    const float u1 = fmaxf(1.0e-7f, word_to_uniform(c[0]));
    const float u2 = word_to_uniform(c[1]);
    const float r = sqrtf(-2.0f * logf(u1));
    dst[col] = r * cosf(6.2831855f * u2) * a.scale;
  }
}

static size_t select_ws_offset(int64_t rows, int64_t n_tiles) {
  return ((size_t)(rows * n_tiles) * sizeof(float) + 255) & ~(size_t)255;
}

// The sampler's workgroups: with enough rows to fill the chip (two workgroups per CU) by
// steps of 1024 threads, as few parts per row as do (a part's first step pays for its
// bound; a part of a very long row has at least 8 steps); with fewer rows one 256-thread
// step per workgroup. us, 256 x 151936, 256 / 1024 threads: T = 0.9 66 / 62, 1.2 79 / 86,
// equal logits 94 / 107, all greedy 29 / 28 (every logit drawn for: 91, and 25 all greedy); 400 rows, T = 0.9 92 /
// 70, 1.2 112 / 120, all greedy 40 / 33 (136, and 33).
// How the sampler takes a call: threads per workgroup and workgroups per row.
struct SamplePlan {
  int threads;
  int64_t parts;
};
// Logits from which a call's workgroups carry their bound over several tiles. Below, one
// 256-thread tile each spreads best; us, 256 threads / 512 threads over two tiles, 400 x
// 151936 (above): T = 0.6 56 / 47, 1.2 112 / 105, half greedy 63 / 63, equal 131 / 140; 640 x
// 151936 79 / 63, 170 / 151, 94 / 89, 201 / 210.
constexpr int64_t SAMPLE_LARGE = 50 << 20;
// Rows of at most 2048 columns: one wavefront each from here on, below 256 threads that draw
// for every logit (sample_short). 8192 x 1000: T = 0.6 18 us, equal logits 34 (36 with 256
// threads); 2048 x 2040, equal logits: 20 against 17.5.
constexpr int64_t SAMPLE_NARROW_ROWS = 4096;

// The columns that a row's chunks may cover: its logits and, where rows are not 16-byte
// aligned, those before it in its first granule.
static int64_t sample_span(int64_t vocab, bool vec) { return vec ? vocab : vocab + 7; }

// Large calls on 2-byte logits: one 1024-thread workgroup per row, whose bound is the row's
// own, where the rows fill the CUs evenly (the last round of rows at least 95 % full);
// elsewhere the CUs with a row more would set the time (640 x 151936, equal logits: 251 us
// against 210), and 512 threads take two tiles each. us, 1024 x 151936, 1024 threads / 512:
// T = 0.6 76 / 98, 1.2 202 / 243, half greedy 138 / 129, equal 333 / 327 (before the last
// shortening of both). Float32 tiles leave room for half the wavefronts there (equal logits
// 390 us against 321 with 256 threads).
static SamplePlan sample_plan(int64_t rows, int64_t vocab, bool vec, bool half) {
  const int64_t span = sample_span(vocab, vec);
  auto tiles = [&](int threads) { return (span + sample_tile(threads) - 1) / sample_tile(threads); };
  if (span <= sample_tile(64) && rows >= SAMPLE_NARROW_ROWS) return SamplePlan{64, 1};
  if (!half || span <= sample_tile(512) || rows * vocab < SAMPLE_LARGE) return SamplePlan{256, tiles(256)};
  DeviceInfo info;
  const int64_t cus = device_info(&info) == FM_OK ? info.cus : 256;
  const int64_t rounds = (rows + cus - 1) / cus;
  if (span > 2 * sample_tile(1024) && 20 * rounds * cus <= 21 * rows) return SamplePlan{1024, 1};
  return SamplePlan{512, (tiles(512) + 1) / 2};
}

static int run_select(const void *logits, int32_t dtype, int64_t rows, int64_t vocab, int64_t row_stride,
                      const float *temps, const uint8_t *greedy, const int64_t *seed, int64_t *out, void *ws,
                      size_t ws_bytes, void *stream) {
  FM_REQUIRE(rows >= 0 && vocab >= 0, "bad sizes");
  if (rows == 0) return FM_OK;
  FM_REQUIRE(vocab > 0, "an empty vocabulary has no argmax");
  FM_REQUIRE(vocab <= INT32_MAX, "vocabulary of %lld above 2^31 - 1", (long long)vocab);
  FM_REQUIRE(rows <= 65535, "at most 65535 rows per call, got %lld", (long long)rows);
  FM_REQUIRE(logits && out && ws, "NULL logits/out/workspace");
  FM_REQUIRE(dtype == LOGITS_BF16 || dtype == LOGITS_F16 || dtype == LOGITS_F32, "unknown logits dtype %d", dtype);
  FM_REQUIRE(row_stride >= vocab, "row stride %lld below the vocabulary %lld", (long long)row_stride,
             (long long)vocab);
  const bool sample = temps != nullptr;
  const int es = dtype == LOGITS_F32 ? 4 : 2;
  const bool vec = (uintptr_t)logits % 16 == 0 && row_stride * es % 16 == 0;
  const SamplePlan plan = sample_plan(rows, vocab, vec, es == 2);
  const int64_t n_tiles = sample ? plan.parts : (vocab + SEL_TILE - 1) / SEL_TILE;
  const size_t need = select_ws_offset(rows, n_tiles) + (size_t)(rows * n_tiles) * sizeof(int32_t);
  if (ws_bytes < need) return fail(FM_ERR_WORKSPACE, "workspace of %zu bytes, %zu needed", ws_bytes, need);
  SelectArgs a{};
  a.logits = (const char *)logits;
  a.row_bytes = row_stride * es;
  a.vocab = vocab;
  a.n_tiles = (int32_t)n_tiles;
  a.vec = vec;
  a.temps = temps;
  a.greedy = greedy;
  a.seed = seed;
  a.best = (float *)ws;
  a.index = (int32_t *)((char *)ws + select_ws_offset(rows, n_tiles));
  hipStream_t s = (hipStream_t)stream;
  const dim3 grid((unsigned)n_tiles, (unsigned)rows);
#define FM_SAMPLE(TY, THREADS, SEVERAL) \
  hipLaunchKernelGGL((sample_parts_kernel<TY, THREADS, SEVERAL>), grid, dim3(THREADS), 0, s, a)
#define FM_SEL(TY)                                                                     \
  do {                                                                                 \
    if (!sample)                                                                       \
      hipLaunchKernelGGL((select_tiles_kernel<TY>), grid, dim3(SEL_THREADS), 0, s, a); \
    else if (plan.threads == 64)                                                       \
      FM_SAMPLE(TY, 64, false);                                                        \
    else if (TY == LOGITS_F32 || plan.threads == 256)                                  \
      FM_SAMPLE(TY, 256, false);                                                       \
    else if (plan.threads == 512)                                                      \
      FM_SAMPLE(TY == LOGITS_F32 ? LOGITS_BF16 : TY, 512, true);                       \
    else                                                                               \
      FM_SAMPLE(TY == LOGITS_F32 ? LOGITS_BF16 : TY, 1024, true);                      \
  } while (0)
  if (dtype == LOGITS_BF16)
    FM_SEL(LOGITS_BF16);
  else if (dtype == LOGITS_F16)
    FM_SEL(LOGITS_F16);
  else
    FM_SEL(LOGITS_F32);
#undef FM_SEL
#undef FM_SAMPLE
  FM_CHECK_HIP(hipGetLastError());
  hipLaunchKernelGGL(select_rows_kernel, dim3((unsigned)rows), dim3(64), 0, s, a.best, a.index, a.n_tiles, out);
  FM_CHECK_HIP(hipGetLastError());
  return FM_OK;
}

}  // namespace fm

using namespace fm;

extern "C" size_t fm_select_workspace_bytes(int64_t rows, int64_t vocab) {
  if (rows <= 0 || vocab <= 0) return 0;
  const int64_t n_tiles = (sample_span(vocab, false) + sample_tile(256) - 1) / sample_tile(256);  // the finest tiling: enough for both
  return select_ws_offset(rows, n_tiles) + (size_t)(rows * n_tiles) * sizeof(int32_t);
}

extern "C" int fm_argmax_rows(const void *logits, int32_t dtype, int64_t rows, int64_t vocab, int64_t row_stride,
                              int64_t *out, void *workspace, size_t workspace_bytes, void *stream) {
  clear_error();
  return run_select(logits, dtype, rows, vocab, row_stride, nullptr, nullptr, nullptr, out, workspace,
                    workspace_bytes, stream);
}

extern "C" int fm_sample_rows(const void *logits, int32_t dtype, int64_t rows, int64_t vocab, int64_t row_stride,
                              const float *temperatures, const uint8_t *greedy, const int64_t *seed, int64_t *out,
                              void *workspace, size_t workspace_bytes, void *stream) {
  clear_error();
  FM_REQUIRE(rows == 0 || (temperatures && greedy && seed), "NULL temperatures/greedy/seed");
  return run_select(logits, dtype, rows, vocab, row_stride, temperatures, greedy, seed, out, workspace,
                    workspace_bytes, stream);
}

extern "C" int fm_seeded_normal(const int64_t *seeds, const void *rows, int32_t rows_int64, const void *positions,
                                int32_t positions_int64, int64_t num_rows, int64_t n_cols, float scale, float *out,
                                int64_t out_row_stride, void *stream) {
  clear_error();
  FM_REQUIRE(num_rows >= 0 && n_cols >= 0, "bad sizes");
  if (num_rows == 0 || n_cols == 0) return FM_OK;
  FM_REQUIRE(seeds && rows && positions && out, "NULL seeds/rows/positions/out");
  FM_REQUIRE(num_rows <= 65535, "at most 65535 rows per call, got %lld", (long long)num_rows);
  FM_REQUIRE(out_row_stride >= n_cols, "output row stride below n_cols");
  NoiseArgs a{seeds, rows, positions, rows_int64 ? 1 : 0, positions_int64 ? 1 : 0, n_cols, out_row_stride, scale, out};
  const dim3 grid((unsigned)((n_cols + NOISE_COLS - 1) / NOISE_COLS), (unsigned)num_rows);
  hipLaunchKernelGGL(seeded_normal_kernel, grid, dim3(256), 0, (hipStream_t)stream, a);
  FM_CHECK_HIP(hipGetLastError());
  return FM_OK;
}
