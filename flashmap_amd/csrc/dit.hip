// The DiT's residual stream between its sublayers (flashmap/modeling_flashmap.py:102-117,
// 185-192): after a sublayer's output y, the gated residual x' = x + gate * y, then the
// next sublayer's time-modulated LayerNorm h = LN(x') * (1 + scale) + shift. The
// reference runs these as about eight eager bf16 ops per sublayer; here one pass per row
// reads x and y once and writes x' and h.
//
// Rounding points are torch's eager bf16 ones: gate * y, x + (gate * y), LN(x'),
// 1 + scale, LN * (1 + scale) and + shift each round to bf16 (each computed in fp32 from
// bf16 operands, products and sums kept apart so nothing contracts into an FMA). LN is
// without affine weights, (x' - mean) * rsqrt(var + eps) with the biased variance, its
// statistics reduced in fp32 over the row (two passes over the row held in registers).
// The statistics' summation order is the only difference from torch's kernel, so x' is
// bit-exact and h agrees up to an occasional one-ulp flip of the LN rounding.
//
// Layout: rows of `dim` bf16 values with a row stride, one wavefront per row; lane l
// holds the 16-byte chunks l, l + 64, ... of its row (coalesced 1 KiB per wavefront
// load). gate, scale and shift are (dim,) vectors shared by every row: the modulations
// depend on the jump's times only. Two variants serve the folded noise read-out of a
// one-jump draft (flashmap/vllm/model.py:915-925): the gate one bf16 scalar per row, and
// x one (dim,) row shared by all rows (row stride 0).
//
// fm_noise_rows, that read-out's row pass: per row of the fp32 noise z (H values) the
// scale bf16(gain * rsqrt(sum_i z_i^2 lambda_i + eps)) and z rounded to bf16 for the
// folded GEMM; one wavefront per row, 16-byte loads.
#include "fm_device.h"
#include "fm_host.h"

namespace fm {

struct AdalnArgs {
  const uint16_t *x;
  const uint16_t *y;  // NULL: no residual, x' = x
  const uint16_t *gate, *scale, *shift;  // scale NULL: no norm
  int32_t gate_rows;  // nonzero: gate holds one value per row
  uint16_t *x_out;  // NULL: x' not stored
  uint16_t *h_out;
  int64_t rows;
  int64_t xs, ys, xos, hs;  // row strides (elements)
  int32_t dim;
  float eps;
};

__device__ __forceinline__ float wave_sum64(float v) {
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) v = __fadd_rn(v, __shfl_xor(v, m, 64));
  return v;
}

template <int NCH>
__global__ __launch_bounds__(256) void adaln_residual_kernel(const AdalnArgs a) {
  const int lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * 4 + wave_id();
  if (row >= a.rows) return;  // wave-uniform
  const int chunks = a.dim >> 3;
  u32x4_t r[NCH];
  float sum = 0.f;
#pragma unroll
  for (int i = 0; i < NCH; ++i) {
    const int c = lane + 64 * i;
    if (c < chunks) {
      const u32x4_t xv = load16(a.x + row * a.xs + 8 * c);
      if (a.y != nullptr) {
        const u32x4_t yv = load16(a.y + row * a.ys + 8 * c);
        u32x4_t gv;
        if (a.gate_rows) {
          const uint32_t gr = a.gate[row];
          const uint32_t g2 = gr | (gr << 16);
          gv = u32x4_t{g2, g2, g2, g2};
        } else {
          gv = load16(a.gate + 8 * c);
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const float lo = __fadd_rn(bf16_lo(xv[q]), round_bf16(__fmul_rn(bf16_lo(gv[q]), bf16_lo(yv[q]))));
          const float hi = __fadd_rn(bf16_hi(xv[q]), round_bf16(__fmul_rn(bf16_hi(gv[q]), bf16_hi(yv[q]))));
          r[i][q] = pack_bf16x2(lo, hi);
        }
      } else {
        r[i] = xv;
      }
#pragma unroll
      for (int q = 0; q < 4; ++q) sum = __fadd_rn(sum, __fadd_rn(bf16_lo(r[i][q]), bf16_hi(r[i][q])));
      if (a.x_out != nullptr) store16(a.x_out + row * a.xos + 8 * c, r[i]);
    }
  }
  if (a.scale == nullptr) return;
  const float n = (float)a.dim;
  const float mean = __fdiv_rn(wave_sum64(sum), n);
  float sq = 0.f;
#pragma unroll
  for (int i = 0; i < NCH; ++i) {
    if (lane + 64 * i < chunks) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const float dl = __fsub_rn(bf16_lo(r[i][q]), mean), dh = __fsub_rn(bf16_hi(r[i][q]), mean);
        sq = __fadd_rn(sq, __fadd_rn(__fmul_rn(dl, dl), __fmul_rn(dh, dh)));
      }
    }
  }
  const float rstd = rsqrtf(__fadd_rn(__fdiv_rn(wave_sum64(sq), n), a.eps));
#pragma unroll
  for (int i = 0; i < NCH; ++i) {
    const int c = lane + 64 * i;
    if (c < chunks) {
      const u32x4_t sv = load16(a.scale + 8 * c);
      const u32x4_t tv = load16(a.shift + 8 * c);
      u32x4_t h;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        float v[2] = {bf16_lo(r[i][q]), bf16_hi(r[i][q])};
        const float s[2] = {bf16_lo(sv[q]), bf16_hi(sv[q])};
        const float t[2] = {bf16_lo(tv[q]), bf16_hi(tv[q])};
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const float ln = round_bf16(__fmul_rn(rstd, __fsub_rn(v[j], mean)));
          const float mod = round_bf16(__fmul_rn(ln, round_bf16(__fadd_rn(1.0f, s[j]))));
          v[j] = __fadd_rn(mod, t[j]);
        }
        h[q] = pack_bf16x2(v[0], v[1]);
      }
      store16(a.h_out + row * a.hs + 8 * c, h);
    }
  }
}

// One wavefront per row of z (fp32, H values): lane l holds the 4-value chunks l, l + 64, ...
template <int NCH>
__global__ __launch_bounds__(256) void noise_rows_kernel(const float *__restrict__ z, int64_t rows, int32_t h,
                                                         int64_t zs, const float *__restrict__ lam, float eps,
                                                         float gain, uint16_t *__restrict__ z16, int64_t z16s,
                                                         uint16_t *__restrict__ scale) {
  const int lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * 4 + wave_id();
  if (row >= rows) return;  // wave-uniform
  const int chunks = h >> 2;
  float acc = 0.f;
#pragma unroll
  for (int i = 0; i < NCH; ++i) {
    const int c = lane + 64 * i;
    if (c < chunks) {
      const f32x4_t v = *reinterpret_cast<const f32x4_t *>(z + row * zs + 4 * c);
      const f32x4_t l = *reinterpret_cast<const f32x4_t *>(lam + 4 * c);
#pragma unroll
      for (int q = 0; q < 4; ++q) acc = __builtin_fmaf(__fmul_rn(v[q], v[q]), l[q], acc);
      *reinterpret_cast<u32x2_t *>(z16 + row * z16s + 4 * c) = u32x2_t{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
    }
  }
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) acc = __fadd_rn(acc, __shfl_xor(acc, m, 64));
  if (lane == 0) {
    const float s = __fmul_rn(gain, rsqrtf(__fadd_rn(acc, eps)));
    scale[row] = (uint16_t)(pack_bf16x2(s, 0.f) & 0xffffu);
  }
}

static bool aligned16(const void *p) { return ((uintptr_t)p & 15) == 0; }

// The several-jump draft's state over the vocabulary (flashmap/vllm/model.py:944-956,
// 1031-1036): softmaxes over rows of up to ~10^5 values. A row goes to `parts` workgroups
// (state_parts); each forms the whole row's statistics (max and sum of exponentials,
// online per thread, merged over the workgroup) and writes its part of the outputs. The
// statistics are taken in one order whatever the part: a row's values do not depend on how
// many rows the call has.
//
// Bound: HBM for a full batch over a whole vocabulary. Few rows are in flight there (one
// 1024-thread workgroup per CU, or two), so that the second read of a row comes from the
// caches: with 256-thread workgroups each of 1024 rows was resident at once, 311 to 622 MB
// between the two reads. The arithmetic stays below the stream: exponentials are exp_neg (9
// issue slots against 18 for expf), the divisions by a row's (or the call's) one divisor take
// its reciprocal once and three operations per element (DivBy; 14 for an IEEE division), the
// products' maximum one product. Measured, 1024 x 151936 (1.56 and 1.24 GB) with 256 threads,
// expf and IEEE divisions / now: update 422 / 281 us, embedding 388 / 260 us (16 chunks held
// spill: 347 us). In parts, 64 rows: update 162 / 42 us, embedding 153 / 38 us.
constexpr int STATE_CHUNKS = 4;  // 4-value chunks in flight per thread
constexpr int STATE_HELD = 8;    // state_embed_rows: chunks per thread kept between the passes

// exp(x) for x <= 0 (0 for -inf, NaN for NaN) to about an ulp: exp2 of the rounded x log2(e),
// corrected by what that rounding left of x. r is NaN only for x = -inf (the result is 0
// already) and NaN (the result is NaN): the max keeps it out of the product. Results below
// 2^-126 are 0 (the hardware's exp2 has no subnormals): for the sums, whose largest term is 1.
__device__ __forceinline__ float exp_neg(float x) {
#pragma clang fp contract(off)  // r is taken from the rounded t
  const float t = x * 1.44269504f;
  const float p = __builtin_amdgcn_exp2f(t);
  const float r = __builtin_fmaf(-t, -1.90465421e-9f, __builtin_fmaf(-t, 0.693147182f, x));
  return __builtin_fmaf(p, fmaxf(r, -0.001f), p);
}

// 2^24 exp(x), for the outputs, whose divisor carries the same factor: exp2's results are
// normal wherever exp(x) is at least a subnormal. The subtraction is exact (u has t's grid
// where it is the smaller of the two, and is within a factor of two of 24 elsewhere).
constexpr float EXP_SCALE = 0x1p24f;
__device__ __forceinline__ float exp_scaled(float x) {
  const float u = __builtin_fmaf(x, 1.44269504f, 24.f);
  const float p = __builtin_amdgcn_exp2f(u);
  const float t = u - 24.f;
  const float r = __builtin_fmaf(-t, -1.90465421e-9f, __builtin_fmaf(-t, 0.693147182f, x));
  return __builtin_fmaf(p, fmaxf(r, -0.001f), p);
}

// a / c by c's correctly rounded reciprocal and one residual step: the rounded quotient
// (4 x 10^6 random numerators over each of six divisors from 26 to 2843: no difference).
struct DivBy {
  float c, y;
  __device__ __forceinline__ explicit DivBy(float c_) : c(c_), y(__fdiv_rn(1.0f, c_)) {}
  __device__ __forceinline__ float operator()(float a) const {
    const float q = a * y;
    return __builtin_fmaf(__builtin_fmaf(-q, c, a), y, q);
  }
  // The same where the quotient may be infinite (the residual is then NaN).
  __device__ __forceinline__ float any(float a) const {
    const float q = a * y, d = __builtin_fmaf(__builtin_fmaf(-q, c, a), y, q);
    return d == d ? d : q;
  }
};

// The exponent of a value: what the product scale * x leaves of the row's max m (a rounded
// product itself) in one rounding, or x - m. The same in the sum and in the outputs, which
// therefore add up to 1 at any scale: at products of 4e6 the max is rounded by up to 0.25,
// and an exponent that rounds the product first differs by a factor of up to 1.28.
template <bool SCALED>
__device__ __forceinline__ float below(float x, float scale, float m) {
  return SCALED ? __builtin_fmaf(x, scale, -m) : x - m;
}

// m starts at the lowest finite value, so that no difference below is inf - inf unless a
// value is +inf (the row is then NaN, as torch has it).
struct RowStats {
  float m, s;  // max and sum of exp(x - m)
  static __device__ __forceinline__ RowStats none() { return RowStats{-3.402823466e38f, 0.f}; }
  __device__ __forceinline__ void raise(float mx) {
    if (mx > m) {
      s *= exp_neg(m - mx);
      m = mx;
    }
  }
  __device__ __forceinline__ void merge(const RowStats &o) {
    const float mx = fmaxf(m, o.m);
    s = s * exp_neg(m - mx) + o.s * exp_neg(o.m - mx);
    m = mx;
  }
};

template <bool SCALED, int N>
__device__ __forceinline__ void add_values(RowStats &st, const float (&x)[N], float scale) {
  // The largest rounded product is the rounded product of the largest value (the smallest
  // for a negative scale).
  float mx = x[0];
  if (SCALED && scale < 0.f) {
#pragma unroll
    for (int q = 1; q < N; ++q) mx = fminf(mx, x[q]);
  } else {
#pragma unroll
    for (int q = 1; q < N; ++q) mx = fmaxf(mx, x[q]);
  }
  st.raise(SCALED ? mx * scale : mx);
  float s = 0.f;
#pragma unroll
  for (int q = 0; q < N; ++q) s += exp_neg(below<SCALED>(x[q], scale, st.m));
  st.s += s;
}

// The workgroup's statistics from each thread's.
template <int THREADS>
__device__ __forceinline__ RowStats block_stats(RowStats st) {
  __shared__ RowStats part[THREADS / 64];
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    st.merge(RowStats{__shfl_xor(st.m, o, 64), __shfl_xor(st.s, o, 64)});
  }
  if ((threadIdx.x & 63) == 0) part[wave_id()] = st;
  __syncthreads();
  RowStats r = part[0];
#pragma unroll
  for (int w = 1; w < THREADS / 64; ++w) r.merge(part[w]);
  return r;
}

// Four consecutive values of a row of float or bf16.
__device__ __forceinline__ f32x4_t load4(const float *p) { return *reinterpret_cast<const f32x4_t *>(p); }
__device__ __forceinline__ f32x4_t load4(const uint16_t *p) {
  const u32x2_t w = *reinterpret_cast<const u32x2_t *>(p);
  return f32x4_t{bf16_lo(w[0]), bf16_hi(w[0]), bf16_lo(w[1]), bf16_hi(w[1])};
}
// Accesses of what the kernel does not touch again. NT: past the caches (non-temporal), so
// that these keep the rows between their two reads; for outputs that would not stay in the
// caches for the next kernel anyway (state_streams).
template <bool NT>
__device__ __forceinline__ f32x4_t load_last(const float *p) {
  return NT ? __builtin_nontemporal_load(reinterpret_cast<const f32x4_t *>(p)) : load4(p);
}
template <bool NT, typename T, typename V>
__device__ __forceinline__ void store_last(T *p, V v) {
  if (NT)
    __builtin_nontemporal_store(v, reinterpret_cast<V *>(p));
  else
    *reinterpret_cast<V *>(p) = v;
}
__device__ __forceinline__ float load1(const float *p) { return *p; }
__device__ __forceinline__ float load1(const uint16_t *p) { return bf16_to_f32(*p); }

// Adds scale * x (SCALED; else x) over the 4-value chunks [from, end) of a row to this
// thread's statistics.
template <int THREADS, bool SCALED, typename T>
__device__ __forceinline__ void add_chunks(RowStats &st, const T *x, int64_t from, int64_t end, float scale) {
  int64_t c = from + threadIdx.x;
  for (; c + (STATE_CHUNKS - 1) * THREADS < end; c += STATE_CHUNKS * THREADS) {
    float e[4 * STATE_CHUNKS];
#pragma unroll
    for (int k = 0; k < STATE_CHUNKS; ++k) {
      const f32x4_t v = load4(x + 4 * (c + k * THREADS));
#pragma unroll
      for (int q = 0; q < 4; ++q) e[4 * k + q] = v[q];
    }
    add_values<SCALED>(st, e, scale);
  }
  for (; c < end; c += THREADS) {
    const f32x4_t v = load4(x + 4 * c);
    const float e[4] = {v[0], v[1], v[2], v[3]};
    add_values<SCALED>(st, e, scale);
  }
}
// ... over the values past a row's last whole chunk (vocab % 4 of them).
template <int THREADS, bool SCALED, typename T>
__device__ __forceinline__ void add_tail(RowStats &st, const T *x, int64_t vocab, float scale) {
  for (int64_t i = (vocab & ~3ll) + threadIdx.x; i < vocab; i += THREADS) {
    const float e[1] = {load1(x + i)};
    add_values<SCALED>(st, e, scale);
  }
}

// This workgroup's part of a row of `chunks` 4-value chunks; the last part also takes the
// values past them.
struct PartOf {
  int64_t first, end;
  bool last;
};
__device__ __forceinline__ PartOf part_of(int64_t chunks) {
  const uint32_t parts = gridDim.y, p = blockIdx.y;  // a power of two
  const int sh = 31 - __builtin_clz(parts);
  return PartOf{chunks * p >> sh, chunks * (p + 1) >> sh, p == parts - 1};
}

// POST: rows r < rows of out (`rows`: the call's, where out begins at this launch's) get bf16(softmax(evidence * state[r])) and rows rows + r
// bf16(state[r]); otherwise out holds the state rows only (one read of the row). A
// workgroup keeps the row's first STATE_HELD chunks per thread in registers between the two
// passes (32768 values of 1024 threads), for the part that begins there; the rest is read
// again from the caches.
template <bool POST, bool NT, int THREADS>
__global__ __launch_bounds__(THREADS) void state_embed_rows_kernel(const float *__restrict__ state,
                                                                         int64_t vocab, int64_t ss, float evidence,
                                                                         uint16_t *__restrict__ out, int64_t os,
                                                                         int64_t rows) {
  const int64_t row = blockIdx.x;
  const float *x = state + row * ss;
  const int64_t chunks = vocab >> 2;
  uint16_t *post = out + row * os, *raw = POST ? out + (rows + row) * os : post;
  const PartOf part = part_of(chunks);
  RowStats t{0.f, 1.f};
  f32x4_t held[STATE_HELD];
  if constexpr (POST) {
    t = RowStats::none();
#pragma unroll
    for (int k = 0; k < STATE_HELD; ++k) {
      const int64_t c = threadIdx.x + k * THREADS;
      held[k] = c < chunks ? load4(x + 4 * c) : f32x4_t{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int k = 0; k < STATE_HELD; k += STATE_CHUNKS) {
      if (threadIdx.x + (k + STATE_CHUNKS - 1) * THREADS < chunks) {
        float e[4 * STATE_CHUNKS];
#pragma unroll
        for (int q = 0; q < 4 * STATE_CHUNKS; ++q) e[q] = held[k + q / 4][q % 4];
        add_values<true>(t, e, evidence);
      } else {
#pragma unroll
        for (int j = k; j < k + STATE_CHUNKS; ++j) {
          if (threadIdx.x + j * THREADS < chunks) {
            const float e[4] = {held[j][0], held[j][1], held[j][2], held[j][3]};
            add_values<true>(t, e, evidence);
          }
        }
      }
    }
    add_chunks<THREADS, true>(t, x, STATE_HELD * THREADS, chunks, evidence);
    add_tail<THREADS, true>(t, x, vocab, evidence);
    t = block_stats<THREADS>(t);
  }
  const DivBy div(t.s * EXP_SCALE);
  auto put = [&](int64_t c, f32x4_t v) {
    if constexpr (POST) {
      float p[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) p[q] = div(exp_scaled(below<true>(v[q], evidence, t.m)));
      store_last<NT>(post + 4 * c, u32x2_t{pack_bf16x2(p[0], p[1]), pack_bf16x2(p[2], p[3])});
    }
    store_last<NT>(raw + 4 * c, u32x2_t{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])});
  };
  int64_t c = part.first + threadIdx.x;
  if constexpr (POST) {
    if (part.first == 0) {
#pragma unroll
      for (int k = 0; k < STATE_HELD; ++k, c += THREADS)
        if (c < part.end) put(c, held[k]);
    }
  }
#pragma unroll 4
  for (; c < part.end; c += THREADS) put(c, load_last<NT>(x + 4 * c));
  if (!part.last) return;
  for (int64_t i = 4 * chunks + threadIdx.x; i < vocab; i += THREADS) {
    if constexpr (POST)
      post[i] = (uint16_t)(pack_bf16x2(div(exp_scaled(below<true>(x[i], evidence, t.m))), 0.f) & 0xffffu);
    raw[i] = (uint16_t)(pack_bf16x2(x[i], 0.f) & 0xffffu);
  }
}

// state[r] = (c_keep * state[r] + c_new * softmax(logits[r])) / c_div in place, logits bf16.
template <bool NT, int THREADS>
__global__ __launch_bounds__(THREADS) void state_update_kernel(float *__restrict__ state, int64_t vocab,
                                                                     int64_t ss, const uint16_t *__restrict__ logits,
                                                                     int64_t ls, float c_keep, float c_new,
                                                                     float c_div) {
  const int64_t row = blockIdx.x;
  float *x = state + row * ss;
  const uint16_t *lg = logits + row * ls;
  const int64_t chunks = vocab >> 2;
  const PartOf part = part_of(chunks);
  RowStats t = RowStats::none();
  add_chunks<THREADS, false>(t, lg, 0, chunks, 1.f);
  add_tail<THREADS, false>(t, lg, vocab, 1.f);
  t = block_stats<THREADS>(t);
  const DivBy div(t.s * EXP_SCALE), scale(c_div);
  auto upd = [&](float s, float l) {
    return scale.any(__builtin_fmaf(c_keep, s, c_new * div(exp_scaled(l - t.m))));
  };
#pragma unroll 4
  for (int64_t c = part.first + threadIdx.x; c < part.end; c += THREADS) {
    const int64_t at = 4 * c;
    const f32x4_t l = load4(lg + at);
    f32x4_t v = load_last<NT>(x + at);
#pragma unroll
    for (int q = 0; q < 4; ++q) v[q] = upd(v[q], l[q]);
    store_last<NT>(x + at, v);
  }
  if (!part.last) return;
  for (int64_t i = 4 * chunks + threadIdx.x; i < vocab; i += THREADS) x[i] = upd(x[i], load1(lg + i));
}

// Whether a call's state rows outgrow the 256 MB of the last cache level. Below that the
// kernels' outputs are found there by whoever reads them next, and the non-temporal
// accesses only cost: the state rows alone at 256 x 151936 (156 MB) 33 us, 42 us with them.
static bool state_streams(int64_t rows, int64_t vocab) { return rows * vocab > (64ll << 20); }

// Workgroups per row, a power of two: doubled while they are no more than the CUs (so 257 rows
// and more are not split on 256 CUs); each part reads the whole row for its statistics again
// (from the caches).
static unsigned state_parts(int64_t rows) {
  DeviceInfo info;
  if (device_info(&info) != FM_OK) return 1;
  unsigned p = 1;
  while (p < 8 && p * rows <= (int64_t)info.cus) p *= 2;
  return p;
}

// Threads per workgroup, by the vocabulary alone (so that the order of a row's sum is). Short
// rows want small workgroups: what a row costs is then its barrier and its one round of loads.
// us, 256 / 512 / 1024 threads, update and embedding: 8192 x 1000 22 / 39 / 95 and 20 / 40 /
// 106; 1024 x 8192 15 / 17 / 23 and 17 / 17 / 24; 1024 x 16384 30 / 30 / 33 and 26 / 27 / 35;
// 1024 x 32000 58 / 58 / 59 and 54 / 50 / 55; 300 x 65536 47 / 45 / 49 and 41 / 44 / 48; 1024
// x 65536 143 / 139 / 136 and 146 / 145 / 127; 1024 x 151936 333 / 321 / 283 and 309 / 289 /
// 260. (Every size with 256 threads, expf and IEEE divisions: 32 and 30, 21 and 18, 38 and 33,
// 71 and 61, 86 and 75, 173 and 164, 422 and 388.)
static int state_threads(int64_t vocab) { return vocab <= 12288 ? 256 : vocab <= 40960 ? 512 : 1024; }

// launch(first row, rows) over slices of a call's rows: a grid counts at most 2^32 - 1 threads.
template <typename F>
static void for_row_slices(int64_t rows, F &&launch) {
  constexpr int64_t SLICE = 1 << 20;
  for (int64_t r = 0; r < rows; r += SLICE) launch(r, (unsigned)(rows - r < SLICE ? rows - r : SLICE));
}

}  // namespace fm

extern "C" int fm_adaln_residual(const void *x, int64_t x_stride, const void *y, int64_t y_stride,
                                 const void *gate, int32_t gate_per_row, const void *scale, const void *shift,
                                 void *x_out, int64_t x_out_stride, void *h_out, int64_t h_out_stride,
                                 int64_t rows, int32_t dim, float eps, void *stream) {
  using namespace fm;
  FM_REQUIRE(rows >= 0 && dim > 0, "bad sizes: rows=%lld dim=%d", (long long)rows, dim);
  if (rows == 0) return FM_OK;
  if (dim % 8 != 0 || dim > 8192)
    return fail(FM_ERR_UNSUPPORTED, "dim %d not supported (a multiple of 8, at most 8192)", dim);
  FM_REQUIRE(x != nullptr, "NULL x");
  FM_REQUIRE(y == nullptr || gate != nullptr, "a residual needs its gate");
  FM_REQUIRE(scale == nullptr || (shift != nullptr && h_out != nullptr), "a norm needs shift and h_out");
  FM_REQUIRE(scale != nullptr || x_out != nullptr, "nothing to write: neither x_out nor a norm");
  const void *ptrs[7] = {x, y, gate, scale, shift, x_out, h_out};
  for (const void *p : ptrs) FM_REQUIRE(p == nullptr || aligned16(p), "tensors must be 16-byte aligned");
  FM_REQUIRE(x_stride % 8 == 0 && y_stride % 8 == 0 && x_out_stride % 8 == 0 && h_out_stride % 8 == 0,
             "row strides must be multiples of 8 elements");
  FM_REQUIRE((x_stride == 0 || x_stride >= dim) && (y == nullptr || y_stride >= dim) &&
                 (x_out == nullptr || x_out_stride >= dim) && (h_out == nullptr || h_out_stride >= dim),
             "row strides must cover a row of %d (x may also be one shared row, stride 0)", dim);
  FM_REQUIRE(x_stride != 0 || x_out != x, "a shared x row cannot be written in place");
  const int64_t blocks = (rows + 3) / 4;
  FM_REQUIRE(blocks < (1ll << 31), "too many rows");
  AdalnArgs a{(const uint16_t *)x,     (const uint16_t *)y,     (const uint16_t *)gate,
              (const uint16_t *)scale, (const uint16_t *)shift, gate_per_row,
              (uint16_t *)x_out,       (uint16_t *)h_out,       rows,
              x_stride,                y_stride,                x_out_stride,
              h_out_stride,            dim,                     eps};
  hipStream_t s = (hipStream_t)stream;
  const int per_lane = (dim / 8 + 63) / 64;
  const dim3 grid((unsigned)blocks), block(256);
  if (per_lane <= 1)
    adaln_residual_kernel<1><<<grid, block, 0, s>>>(a);
  else if (per_lane <= 2)
    adaln_residual_kernel<2><<<grid, block, 0, s>>>(a);
  else if (per_lane <= 4)
    adaln_residual_kernel<4><<<grid, block, 0, s>>>(a);
  else if (per_lane <= 8)
    adaln_residual_kernel<8><<<grid, block, 0, s>>>(a);
  else
    adaln_residual_kernel<16><<<grid, block, 0, s>>>(a);
  FM_CHECK_HIP(hipGetLastError());
  return FM_OK;
}

extern "C" int fm_noise_rows(const float *z, int64_t rows, int32_t hidden, int64_t z_stride, const float *eigvals,
                             float eps, float gain, void *z_bf16, int64_t z_bf16_stride, void *scale,
                             void *stream) {
  using namespace fm;
  FM_REQUIRE(rows >= 0 && hidden > 0, "bad sizes: rows=%lld hidden=%d", (long long)rows, hidden);
  if (rows == 0) return FM_OK;
  if (hidden % 4 != 0 || hidden > 16384)
    return fail(FM_ERR_UNSUPPORTED, "hidden %d not supported (a multiple of 4, at most 16384)", hidden);
  FM_REQUIRE(z && eigvals && z_bf16 && scale, "NULL tensor pointer");
  FM_REQUIRE(aligned16(z) && aligned16(eigvals) && ((uintptr_t)z_bf16 & 7) == 0,
             "z / eigvals must be 16-byte aligned, z_bf16 8-byte aligned");
  FM_REQUIRE(z_stride % 4 == 0 && z_stride >= hidden && z_bf16_stride % 4 == 0 && z_bf16_stride >= hidden,
             "row strides must be multiples of 4 covering a row");
  const int64_t blocks = (rows + 3) / 4;
  FM_REQUIRE(blocks < (1ll << 31), "too many rows");
  hipStream_t s = (hipStream_t)stream;
  const int per_lane = (hidden / 4 + 63) / 64;
  const dim3 grid((unsigned)blocks), block(256);
  uint16_t *zo = (uint16_t *)z_bf16, *so = (uint16_t *)scale;
  if (per_lane <= 8)
    noise_rows_kernel<8><<<grid, block, 0, s>>>(z, rows, hidden, z_stride, eigvals, eps, gain, zo, z_bf16_stride, so);
  else if (per_lane <= 16)
    noise_rows_kernel<16><<<grid, block, 0, s>>>(z, rows, hidden, z_stride, eigvals, eps, gain, zo, z_bf16_stride, so);
  else
    noise_rows_kernel<64><<<grid, block, 0, s>>>(z, rows, hidden, z_stride, eigvals, eps, gain, zo, z_bf16_stride, so);
  FM_CHECK_HIP(hipGetLastError());
  return FM_OK;
}

extern "C" int fm_state_embed_rows(const float *state, int64_t rows, int64_t vocab, int64_t state_stride,
                                   float evidence, int32_t posterior, void *out, int64_t out_stride, void *stream) {
  using namespace fm;
  FM_REQUIRE(rows >= 0 && vocab > 0, "bad sizes: rows=%lld vocab=%lld", (long long)rows, (long long)vocab);
  if (rows == 0) return FM_OK;
  FM_REQUIRE(state && out, "NULL tensor pointer");
  FM_REQUIRE(rows < (1ll << 31), "too many rows");
  FM_REQUIRE(aligned16(state) && state_stride % 4 == 0 && state_stride >= vocab,
             "state must be 16-byte aligned with a row stride that is a multiple of 4 covering a row");
  FM_REQUIRE(((uintptr_t)out & 7) == 0 && out_stride % 4 == 0 && out_stride >= vocab,
             "out must be 8-byte aligned with a row stride that is a multiple of 4 covering a row");
  const bool nt = state_streams(rows, vocab);
  auto run = [&](auto *kernel, int threads, unsigned parts) {
    for_row_slices(rows, [&](int64_t first, unsigned n) {
      kernel<<<dim3(n, parts), dim3(threads), 0, (hipStream_t)stream>>>(
          state + first * state_stride, vocab, state_stride, evidence, (uint16_t *)out + first * out_stride,
          out_stride, rows);
    });
  };
#define FM_EMBED(THREADS) \
  run(nt ? state_embed_rows_kernel<true, true, THREADS> : state_embed_rows_kernel<true, false, THREADS>, THREADS, parts)
  const int threads = state_threads(vocab);
  const unsigned parts = state_parts(rows);
  // The state rows alone are a copy: 1024 threads where they stream (1024 x 151936 171 us, 175
  // with 256), 256 below (300 x 151936 54 us, 57 with 1024; 8192 x 1000 8.2 and 11.2 us), in
  // half as many parts (256 x 151936 33.9 us, 34.9 in two).
  if (!posterior && nt)
    run(state_embed_rows_kernel<false, true, 1024>, 1024, 1);
  else if (!posterior)
    run(state_embed_rows_kernel<false, false, 256>, 256, state_parts(2 * rows));
  else if (threads == 256)
    FM_EMBED(256);
  else if (threads == 512)
    FM_EMBED(512);
  else
    FM_EMBED(1024);
#undef FM_EMBED
  FM_CHECK_HIP(hipGetLastError());
  return FM_OK;
}

extern "C" int fm_state_update(float *state, int64_t rows, int64_t vocab, int64_t state_stride, const void *logits,
                               int64_t logits_stride, double start, double end, void *stream) {
  using namespace fm;
  FM_REQUIRE(rows >= 0 && vocab > 0, "bad sizes: rows=%lld vocab=%lld", (long long)rows, (long long)vocab);
  if (rows == 0) return FM_OK;
  FM_REQUIRE(state && logits, "NULL tensor pointer");
  FM_REQUIRE(rows < (1ll << 31), "too many rows");
  FM_REQUIRE(start < 1.0 && end >= start, "jump times must satisfy start <= end, start < 1 (got %g, %g)", start, end);
  FM_REQUIRE(aligned16(state) && state_stride % 4 == 0 && state_stride >= vocab,
             "state must be 16-byte aligned with a row stride that is a multiple of 4 covering a row");
  FM_REQUIRE(((uintptr_t)logits & 7) == 0 && logits_stride % 4 == 0 && logits_stride >= vocab,
             "logits must be 8-byte aligned with a row stride that is a multiple of 4 covering a row");
  // The scalars as torch takes Python floats into a float32 op: computed in double, then
  // rounded to float.
  const float c_keep = (float)(1.0 - end), c_new = (float)(end - start), c_div = (float)(1.0 - start);
  const bool nt = state_streams(rows, vocab);
  const unsigned parts = state_parts(rows);
  auto run = [&](auto *kernel, int threads) {
    for_row_slices(rows, [&](int64_t first, unsigned n) {
      kernel<<<dim3(n, parts), dim3(threads), 0, (hipStream_t)stream>>>(
          state + first * state_stride, vocab, state_stride, (const uint16_t *)logits + first * logits_stride,
          logits_stride, c_keep, c_new, c_div);
    });
  };
#define FM_UPDATE(THREADS) run(nt ? state_update_kernel<true, THREADS> : state_update_kernel<false, THREADS>, THREADS)
  const int threads = state_threads(vocab);
  if (threads == 256)
    FM_UPDATE(256);
  else if (threads == 512)
    FM_UPDATE(512);
  else
    FM_UPDATE(1024);
#undef FM_UPDATE
  FM_CHECK_HIP(hipGetLastError());
  return FM_OK;
}
