// Token sampler: temperature, top-p filter and one draw per row in one launch, without sorting the row.
// Follows parrot/engine/builtin/models/sampler.py:19-66:
//   :33-40  logits / temperature, the quotient rounded to the logits' element type (in-place division);
//   :43-56  a token is dropped when the probability mass of the tokens sorted before it (descending) exceeds
//           top_p -- the most likely token always stays, and so does the token on which the mass crosses top_p;
//   :63-64  soft-max of the surviving logits, one token drawn from it.
// The reference sorts every row twice (sort, then arg-sort of the permutation) to apply the filter.  Here the
// filter is a threshold: with e_i = exp(x_i - max) and G(t) = sum of e_j over e_j > t, token i stays iff
// G(e_i) + (its rank among equal values) * e_i <= top_p * sum(e).  G is monotone, so the smallest surviving value
// is found by a search over ordered bit patterns.  Equal values are ranked by ascending token id.
// The draw is the inverse-CDF draw over ascending token ids from a uniform number the caller passes, so the
// result is a function of the inputs (the reference draws through torch.multinomial's own random stream).
//
// One workgroup of 1024 lanes per row.  Two kernels, the same e values:
//   sample_rows_kernel   rows on the 16-byte grid of up to 57,344 tokens: the row lives in registers, the cut
//                        comes from histograms of the mass over the bit patterns of e (16-bit rows of few
//                        distinct values, rows with NaN or infinite logits: from the bisection);
//   sample_top_p_kernel  any other row: e values in LDS up to 36 K tokens, longer rows are re-read and
//                        re-exponentiated in every pass (they sit in L2; slower); the cut comes from a bisection
//                        over the patterns of the element type, a compare-and-add over the row per bit.
// Histogram sums are whole numbers (atomic order does not matter), float sums are taken in a fixed order (per-lane
// partial sums, a wave tree, then the sixteen wave sums in sequence): the same tokens on every run.  The histograms'
// masses are exact, the bisection's carry the rounding of fp32 sums (a few 1e-7 of the row's mass): where top_p falls
// that close to the mass before a token, the two can differ by that token, and so can the two kernels (and with them
// ph_sample_top_p and ph_top_p_probs, which takes the second).
#include <type_traits>

#include "common.hpp"

namespace ph {

constexpr int kSampThreads = 1024;
constexpr int kSampWaves = kSampThreads / kWave;
constexpr int kSampLdsFloats = 36 * 1024;

template <typename E>
struct Logit {  // 16-bit element types
  static constexpr int kBytes = 2;
  static __device__ __forceinline__ float load(const void* row, int i) {
    return Elem<E>::one(static_cast<const uint16_t*>(row)[i]);
  }
  static __device__ __forceinline__ float round(float f) { return rnd<E>(f); }
  static __device__ __forceinline__ void unpack(const u32x4 raw, float* x) {  // 8 elements
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      x[2 * j] = Elem<E>::lo(raw[j]);
      x[2 * j + 1] = Elem<E>::hi(raw[j]);
    }
  }
};
template <>
struct Logit<F32> {
  static constexpr int kBytes = 4;
  static __device__ __forceinline__ void unpack(const u32x4 raw, float* x) {  // 4 elements
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint32_t w = raw[j];  // a copy: the cast below is applied to a plain scalar, not to a vector element
      x[j] = __builtin_bit_cast(float, w);
    }
  }
  static __device__ __forceinline__ float load(const void* row, int i) { return static_cast<const float*>(row)[i]; }
  static __device__ __forceinline__ float round(float f) { return f; }
};
// low bits of the fp32 pattern that are zero for every value of the element type
template <typename E> constexpr int key_shift();
template <> constexpr int key_shift<F16>() { return 13; }
template <> constexpr int key_shift<BF16>() { return 16; }
template <> constexpr int key_shift<F32>() { return 0; }

// order-preserving map float -> unsigned (shifted down by SH), and back to the float of a key
template <int SH>
__device__ __forceinline__ uint32_t to_key(float f) {
  uint32_t b = __builtin_bit_cast(uint32_t, f);
  b ^= (b >> 31) ? 0xffffffffu : 0x80000000u;
  return b >> SH;
}
template <int SH>
__device__ __forceinline__ float from_key(uint32_t ks) {
  const uint32_t k = ks << SH;
  const uint32_t b = (k >> 31) ? (k ^ 0x80000000u) : ~(k | ((1u << SH) - 1u));
  return __builtin_bit_cast(float, b);
}

struct SampShared {
  float red[2][kSampWaves];
  float fpart[kSampWaves];
  int ipart[kSampWaves];
  int found, found_after, last;
  int share[kSampWaves];  // sample_rows_kernel: equal values a wave saw
};

struct SampArgs {
  const void* logits;
  int64_t row_stride;  // elements
  const float* temperature;
  const float* top_p;
  const float* uniform;
  int64_t* out;
  int V;
  float* probs;          // set: no draw, the filtered and renormalised probabilities of every row go here
  int64_t probs_stride;  // floats between rows
};

template <typename E, bool LDSX>
__global__ __launch_bounds__(kSampThreads) void sample_top_p_kernel(const SampArgs a) {
  extern __shared__ __attribute__((aligned(16))) float xs[];
  __shared__ SampShared sh;
  constexpr int SH = key_shift<E>();
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  const int64_t row = blockIdx.x;
  const int V = a.V;
  const void* lrow = static_cast<const char*>(a.logits) + row * a.row_stride * Logit<E>::kBytes;
  float T = a.temperature ? a.temperature[row] : 1.f;
  float p = a.top_p ? a.top_p[row] : 1.f;
  if (!(T > 0.f)) {  // the limit of a vanishing temperature: the most likely token
    T = 1.f;
    p = 0.f;
  }
  if (t == 0) {
    sh.found = INT_MAX;
    sh.last = -1;
  }
  int par = 0;
  // block-wide reductions; the two buffers alternate so that one barrier per reduction is enough
  auto block_sum = [&](float v) {
    v = group_sum<64>(v);
    if (lane == 0) sh.red[par][w] = v;
    __syncthreads();
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < kSampWaves; ++i) s += sh.red[par][i];
    par ^= 1;
    return s;
  };
  auto block_max = [&](float v) {
    v = group_max<64>(v);
    if (lane == 0) sh.red[par][w] = v;
    __syncthreads();
    float s = sh.red[par][0];
#pragma unroll
    for (int i = 1; i < kSampWaves; ++i) s = fmaxf(s, sh.red[par][i]);
    par ^= 1;
    return s;
  };
  auto fresh = [&](int i) {
    float l = Logit<E>::load(lrow, i);
    if (T != 1.f) l = Logit<E>::round(__fdiv_rn(l, T));
    return l;
  };

  float m = -INFINITY;
  for (int i = t; i < V; i += kSampThreads) {
    const float x = fresh(i);
    if (LDSX) xs[i] = x;
    m = fmaxf(m, x);
  }
  m = block_max(m);
  if (!(m > -INFINITY && m < INFINITY)) m = 0.f;
  // e_i = exp(x_i - max): computed once and kept in LDS (each lane rewrites the slots it filled itself); every
  // later pass, the equal-value ranking included, works on e alone
  float z = 0.f;
  for (int i = t; i < V; i += kSampThreads) {
    const float e = expf((LDSX ? xs[i] : fresh(i)) - m);
    if (LDSX) xs[i] = e;
    z += e;
  }
  z = block_sum(z);  // and its barrier publishes the e values
  auto e_at = [&](int i) { return LDSX ? xs[i] : expf(fresh(i) - m); };

  // smallest surviving e `thr`, the mass above it, and how many tokens equal to it survive
  float thr = -1.f;  // no filter: everything is above
  int n_equal = INT_MAX;
  if (p < 1.f) {
    const float target = fmaxf(p, 0.f) * z;
    uint32_t lo = to_key<SH>(-INFINITY), hi = to_key<SH>(m);
    float g_hi = 0.f;
    while (lo < hi) {  // lo, hi and g are the same in every lane
      const uint32_t mid = lo + ((hi - lo) >> 1);
      const float cut = expf(from_key<SH>(mid) - m);
      float g = 0.f;
      for (int i = t; i < V; i += kSampThreads) {
        const float e = e_at(i);
        g += e > cut ? e : 0.f;
      }
      g = block_sum(g);
      if (g <= target) {
        hi = mid;
        g_hi = g;
      } else {
        lo = mid + 1;
      }
    }
    thr = expf(from_key<SH>(hi) - m);
    if (thr > 0.f) {
      const float r = floorf((target - g_hi) / thr);
      n_equal = r >= 2.0e9f ? INT_MAX : max((int)r + 1, 1);
    }
  }

  // last pass: every lane owns a run of consecutive token ids (odd length: conflict-free in LDS)
  const int per = ((V + kSampThreads - 1) / kSampThreads) | 1;
  const int b0 = min(t * per, V), b1 = min(b0 + per, V);
  int eq = 0;
  for (int i = b0; i < b1; ++i) eq += e_at(i) == thr ? 1 : 0;
  int inc = eq;  // rank of this lane's first equal token = equal tokens in the lanes before
#pragma unroll
  for (int d = 1; d < kWave; d <<= 1) {
    const int up = __shfl_up(inc, d, kWave);
    if (lane >= d) inc += up;
  }
  if (lane == kWave - 1) sh.ipart[w] = inc;
  __syncthreads();
  int rank0 = inc - eq;
  for (int i = 0; i < w; ++i) rank0 += sh.ipart[i];

  auto walk = [&](auto&& visit) {  // visit(i, e) for every surviving token of this lane's run, in id order
    int rank = rank0;
    for (int i = b0; i < b1; ++i) {
      const float e = e_at(i);
      const bool keep = e > thr || (e == thr && rank++ < n_equal);
      if (keep) visit(i, e);
    }
  };
  float s = 0.f;
  walk([&](int, float e) { s += e; });
  float finc = s;
#pragma unroll
  for (int d = 1; d < kWave; d <<= 1) {
    const float up = __shfl_up(finc, d, kWave);
    if (lane >= d) finc += up;
  }
  if (lane == kWave - 1) sh.fpart[w] = finc;
  __syncthreads();
  float base = 0.f, kept = 0.f;
  for (int i = 0; i < kSampWaves; ++i) {
    if (i == w) base = kept;
    kept += sh.fpart[i];
  }
  base += finc - s;
  if (a.probs) {  // the distribution itself instead of a draw from it: zero for dropped tokens, e / (kept mass) else
    float* prow = a.probs + row * a.probs_stride;
    const float inv = 1.f / kept;
    for (int i = b0; i < b1; ++i) prow[i] = 0.f;
    walk([&](int i, float e) { prow[i] = e * inv; });
    return;
  }
  const float goal = a.uniform[row] * kept;
  int found = INT_MAX, last = -1;
  float running = base;
  walk([&](int i, float e) {
    running += e;
    if (e > 0.f) last = i;
    if (running > goal && found == INT_MAX) found = i;
  });
  if (found != INT_MAX) atomicMin(&sh.found, found);
  if (last >= 0) atomicMax(&sh.last, last);
  __syncthreads();
  if (t == 0) {
    // rounding can leave the goal a hair above the last partial sum: then the last surviving token
    const int id = sh.found != INT_MAX ? sh.found : max(sh.last, 0);
    a.out[row] = id;
  }
}

// x / T rounded to nearest for many x and one T: r = 1 / T rounded to nearest, one Newton correction of x * r, exact
// while nothing leaves the normal range; 3 instructions in place of a division's 10.
__device__ __forceinline__ bool quotient_by_reciprocal(float T) { return T >= 0x1p-40f && T <= 0x1p40f; }
template <typename E>
__device__ __forceinline__ float div_by(float x, float T, float r) {
  const float q = x * r, c = __builtin_fmaf(__builtin_fmaf(-q, T, x), r, q);
  // infinite logits; an fp16 quotient cannot become infinite otherwise, and one instruction tells
  if (std::is_same<E, F16>::value) return __builtin_amdgcn_div_fixupf(c, T, x);
  return __builtin_fabsf(q) < INFINITY ? c : q;
}
// N quotients x / T, rounded to the element type
template <typename E, int N>
__device__ __forceinline__ void divide(float (&x)[N], float T, float r, bool by_r) {
  if (!by_r) {
#pragma unroll
    for (int j = 0; j < N; ++j) x[j] = Logit<E>::round(__fdiv_rn(x[j], T));
    return;
  }
  if constexpr (Logit<E>::kBytes == 2) {
#pragma unroll
    for (int j = 0; j < N; j += 2) {
      const uint32_t two = pack2<E>(div_by<E>(x[j], T, r), div_by<E>(x[j + 1], T, r));
      x[j] = Elem<E>::lo(two);
      x[j + 1] = Elem<E>::hi(two);
    }
  } else {
#pragma unroll
    for (int j = 0; j < N; ++j) x[j] = div_by<E>(x[j], T, r);
  }
}

// Histograms of the mass over the bit pattern of e: 32 bins per power of two, then 8 bits inside the bin the mass
// crosses its target in, then, where that finer bin holds more than one value, the last 10 bits.  Values of one coarse
// bin differ in the low 18 bits of their mantissas only, so a bin takes the tokens' count (from bit 40 up) and the sum
// of those bits: whole numbers, one add per token.  Masses of different bins are compared in units of 2^-46 (a row's
// mass stays below 2^62), inside a bin in mantissas.
typedef unsigned long long mass_t;
constexpr int kHistShift = 18, kHistFine = 8, kHistLast = kHistShift - kHistFine, kHistCount = 40;
constexpr int kHistBins = 2048;  // the bins 2048 .. 4095 of the pattern: from below kHistLeast to beyond e == 1
constexpr uint32_t kHistLeast = 0x21800000u;  // 2^-60: less is no mass
constexpr int kHistFirst = kHistLeast >> kHistShift;  // the bins below hold what is no mass
static_assert(kHistFirst >= kHistBins + kWave && (kHistLeast & ((1u << kHistShift) - 1)) == 0 &&
                  (0x3f800000 >> kHistShift) < 2 * kHistBins && kHistBins == 2 * kSampThreads,
              "two bins per lane");
__device__ __forceinline__ uint32_t mantissa(uint32_t bits) { return (bits & 0x7fffffu) | 0x800000u; }
__device__ __forceinline__ mass_t hist_entry(uint32_t bits) {
  return ((mass_t)1 << kHistCount) | (bits & ((1u << kHistShift) - 1));
}
// Sum of the mantissas of a coarse bin.  (The count times the leading bits as a whole, a product of two 24-bit numbers,
// is miscompiled by this toolchain: it loses the mask of the leading bits.)
__device__ __forceinline__ mass_t hist_mantissas(mass_t entry, uint32_t bin) {
  const uint32_t count = (uint32_t)(entry >> kHistCount);
  return ((mass_t)count << 23) + ((mass_t)(count * (bin & ((1u << (23 - kHistShift)) - 1))) << kHistShift) +
         (entry & (((mass_t)1 << kHistCount) - 1));
}
__device__ __forceinline__ int mass_shift(uint32_t bin) {  // mantissas of a coarse bin << this = units of 2^-46
  return (int)(bin >> (23 - kHistShift)) - (127 - 23);
}
__device__ __forceinline__ mass_t* hist_slot(mass_t* coarse, uint32_t bits) {  // (a pattern of no bin is masked into one)
  return reinterpret_cast<mass_t*>(reinterpret_cast<char*>(coarse) +
                                   ((bits >> (kHistShift - 3)) & ((kHistBins - 1) * sizeof(mass_t))));
}
// Inclusive sum over the lanes, in registers (whole numbers: any order gives the same).
template <int CTRL, int ROWS>
__device__ __forceinline__ mass_t mass_from(mass_t v) {
  const int lo = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)v, CTRL, ROWS, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)(v >> 32), CTRL, ROWS, 0xf, false);
  return ((mass_t)(uint32_t)hi << 32) | (uint32_t)lo;
}
__device__ __forceinline__ mass_t row_prefix_mass(mass_t v) {  // over each row of 16 lanes
  v += mass_from<0x111, 0xf>(v);  // row_shr 1, 2, 4, 8
  v += mass_from<0x112, 0xf>(v);
  v += mass_from<0x114, 0xf>(v);
  v += mass_from<0x118, 0xf>(v);
  return v;
}
__device__ __forceinline__ mass_t wave_prefix_mass(mass_t v) {
  v = row_prefix_mass(v);
  v += mass_from<0x142, 0xa>(v);  // row_bcast 15 into rows 1 and 3
  v += mass_from<0x143, 0xc>(v);  // row_bcast 31 into rows 2 and 3
  return v;
}
__device__ __forceinline__ mass_t lane_mass(mass_t v, int lane) {  // the value of one lane
  return ((mass_t)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(v >> 32), lane) << 32) |
         (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)v, lane);
}
// a / b for a < 2^40 and 2^23 <= b < 2^24: a quotient that is no whole number is further than 2^-24 from one, the
// division's error below 2^-35
__device__ __forceinline__ int count_of(mass_t a, uint32_t b) { return (int)((double)a / (double)b); }

struct SampHist {
  alignas(16) mass_t coarse[kHistBins];
  mass_t fine[1 << kHistFine];
  uint32_t least[1 << kHistFine], most[1 << kHistFine];  // of the patterns in a fine bin
  mass_t last[1 << kHistLast];
  mass_t wave_mass[kSampWaves];
  mass_t goal;     // what the bins still in question may hold above the cut, in mantissas
  uint32_t bin;    // the bin the mass crosses the target in
  uint32_t thr;    // bit pattern of the smallest surviving e (0: not known yet) ...
  int n_equal;     // ... how many tokens of that value survive
  int equal;       // ... and how many there are
};

// One wave looks through the bins of a level, from the top down, for the one the mass crosses the goal in: bins[],
// BITS of them, whose leading bits are `top`.
template <int BITS>
__device__ __forceinline__ void find_in_level(SampHist& hist, const mass_t* level, uint32_t top, int lane, bool last) {
  constexpr int kPer = (1 << BITS) / kWave;
  mass_t bins[kPer], sum = 0;
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    bins[i] = level[(1 << BITS) - 1 - (kPer * lane + i)];
    sum += bins[i];
  }
  const mass_t goal = hist.goal;
  mass_t at = wave_prefix_mass(sum) - sum;
  if (at <= goal && goal < at + sum) {  // one lane
    mass_t in_bin = 0;
    int bin = 0;
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      if (in_bin == 0 && goal < at + bins[i]) {
        in_bin = bins[i];
        bin = (1 << BITS) - 1 - (kPer * lane + i);
      }
      if (in_bin == 0) at += bins[i];
    }
    uint32_t b = (top << BITS) | bin;
    bool one = true;  // one value in the bin
    if (!last) {
      one = hist.least[bin] == hist.most[bin];
      b = one ? hist.least[bin] : b;
    }
    if (one) {
      hist.n_equal = count_of(goal - at, mantissa(b)) + 1;
      hist.equal = count_of(in_bin, mantissa(b));
      hist.thr = b;
    } else {
      hist.goal = goal - at;
      hist.bin = b;
    }
  }
}

// Rows that fit the register file: 16-byte aligned rows of up to 1024 * kSampRegFloats tokens.  Lane t owns the
// 16-byte chunks t, t + 1024, t + 2048, ... of the row (K "rounds" of 1024 chunks); the row is read once, the
// exponentials are taken once, and every later pass is compares and adds on registers.  Token-id order is
// (round, lane, position in the chunk), so the two places that need it -- ranking equal values at the cut and
// the cumulative sum of the draw -- take one batched reduction over the rounds to find the round in which the
// count / the sum crosses, and one scan over the lanes inside that round.
// Bound by vector issue on one compute unit per row and by a chain of ten reductions over the workgroup.  64 rows of
// 32,000 logits, top-p 0.9, fp16 / fp32: 16.0 / 14.6 us.  It was 24.6 / 58 us with one round's load awaited before the
// next was requested, reductions through LDS shuffles, the top-p cut always from three levels, equal values counted lane
// by lane, the uniform number fetched at the draw, and fp32 rows in scratch memory; by bisection alone 37.7 us.  About
// 29 thousand cycles in fp16, read between the phases, whose loads and LDS adds may end in the next one: request 2.4,
// quotients and maximum 5.7, exponentials and coarse bins 4.1, cut 11.3, draw 5.6.
// FLOATS: tokens a lane holds, 32 or kSampRegFloats: the passes are unrolled over them (rows of up to 32,768 tokens
// fetch three fifths of the instructions).
constexpr int kSampRegFloats = 56;
constexpr int kSampShortFloats = 32;

template <typename E, int FLOATS>
__global__ __launch_bounds__(kSampThreads) void sample_rows_kernel(const SampArgs a) {
  constexpr int N = 16 / Logit<E>::kBytes;  // tokens per chunk
  constexpr int K = FLOATS / N;             // chunks per lane
  constexpr int SH = key_shift<E>();
  __shared__ SampShared sh;
  __shared__ SampHist hist;
  __shared__ __attribute__((aligned(16))) float fred[K][kSampWaves];
  __shared__ int ired[K * kSampWaves];
  const int t = threadIdx.x, lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);
  const int64_t row = blockIdx.x;
  const int V = a.V;
  const char* lrow = static_cast<const char*>(a.logits) + row * a.row_stride * Logit<E>::kBytes;

  // the whole row is requested before anything waits for it; chunks that are not whole read the first one instead
  const int chunks = (V + N - 1) / N, whole = V / N;
  const int rounds = (chunks + kSampThreads - 1) / kSampThreads;  // rounds that hold tokens; the rest stay zero
  u32x4 raw[K];
  if (whole > 0) {
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int c = t + k * kSampThreads;
      if (k < rounds) raw[k] = ld16(lrow + (int64_t)(c < whole ? c : 0) * 16);
    }
  }
  if (t == 0) {
    sh.found = INT_MAX;
    sh.found_after = INT_MAX;
    sh.last = -1;
    hist.thr = 0;
  }
  reinterpret_cast<u32x4*>(hist.coarse)[t] = u32x4{0, 0, 0, 0};
  if (t < 1 << kHistFine) {
    hist.fine[t] = 0;
    hist.least[t] = 0xffffffffu;
    hist.most[t] = 0;
  }
  hist.last[t] = 0;
  static_assert(1 << kHistLast == kSampThreads, "one bin of the last level per lane");
  float T = a.temperature ? a.temperature[row] : 1.f;
  float p = a.top_p ? a.top_p[row] : 1.f;
  const float uniform = a.uniform[row];
  if (!(T > 0.f)) {
    T = 1.f;
    p = 0.f;
  }
  const bool filter = p < 1.f;

  int par = 0;
  auto block_sum = [&](float v) {
    v = group_sum<64>(v);
    if (lane == 0) sh.red[par][w] = v;
    __syncthreads();
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < kSampWaves; ++i) s += sh.red[par][i];
    par ^= 1;
    return s;
  };

  auto block_maximum = [&](float v) {
    v = wave_maximum(v);
    if (lane == 0) sh.red[par][w] = v;
    __syncthreads();
    float s = sh.red[par][0];
#pragma unroll
    for (int i = 1; i < kSampWaves; ++i) s = __builtin_elementwise_maximum(s, sh.red[par][i]);
    par ^= 1;
    return s;
  };

  float e[K][N];
#pragma unroll
  for (int k = 0; k < K; ++k) {
    if (k >= rounds) {
#pragma unroll
      for (int j = 0; j < N; ++j) e[k][j] = 0.f;
      continue;
    }
    const int c = t + k * kSampThreads;
    if (whole > 0) Logit<E>::unpack(raw[k], e[k]);
    if (k == rounds - 1) {  // the row's last, partial chunk, and places past the row
      if (c >= whole) {
#pragma unroll
        for (int j = 0; j < N; ++j) e[k][j] = -INFINITY;
        if (c * N < V) {
#pragma unroll
          for (int j = 0; j < N - 1; ++j)
            if (c * N + j < V) e[k][j] = Logit<E>::load(lrow, c * N + j);
        }
      }
    }
  }
  if (T != 1.f) {
    const bool by_r = quotient_by_reciprocal(T);
    const float r = __fdiv_rn(1.f, T);
#pragma unroll
    for (int k = 0; k < K; ++k) {
      if (k >= rounds) break;
      divide<E>(e[k], T, r, by_r);
    }
  }
  float m = -INFINITY;
#pragma unroll
  for (int k = 0; k < K; ++k) {
    if (k >= rounds) break;
#pragma unroll
    for (int j = 0; j < N; ++j) m = __builtin_elementwise_maximum(m, e[k][j]);
  }
  m = wave_maximum(m);
  // Adds of a wave to one address are taken one lane after the other, so a row of few distinct values (equal logits, a
  // high temperature) makes the histograms slow.  Every wave compares one token per chunk with lane 0's: the share in its
  // bin (by distance, half a bin's width) and twice the share of its value.  From one half on the row goes to the
  // bisection.  64 rows of 32,000 fp16 logits, histograms and bisection: all equal 119 and 15.8 us, two values at random
  // 68 and 17, four 43.8 and 38.0, five 37.4 and 36.9, normal logits of deviation 0.005 44.5 and 37.3; eight values (share
  // 0.38) 30.7 and 37.2, deviation 0.02 29.1 and 37.1, deviation 4 15.8 and 35.2 (16.0 with the look).  32-bit logits take
  // the histograms whatever they hold: all equal 99.6 us against 17, but from four values on 45 against 52, deviation 4
  // 14.6 against 48.
  constexpr bool kLooks = Logit<E>::kBytes == 2;
  constexpr float kNoMass = 41.5f;  // this far below the maximum a token is no mass (kHistLeast)
  if (kLooks && filter) {
    int share = 0;
#pragma unroll
    for (int k = 0; k < K; ++k) {
      if (k >= rounds) break;
      const float x = e[k][0];
      const float first = __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, x)));
      if (first > m - kNoMass)  // m: of this wave
        share += __builtin_popcountll(__builtin_amdgcn_ballot_w64(__builtin_fabsf(x - first) < 0.011f)) +
                 2 * __builtin_popcountll(__builtin_amdgcn_ballot_w64(x == first));
    }
    if (lane == 0) sh.share[w] = share;
  }
  if (lane == 0) sh.red[par][w] = m;
  __syncthreads();
  m = sh.red[par][0];
#pragma unroll
  for (int i = 1; i < kSampWaves; ++i) m = __builtin_elementwise_maximum(m, sh.red[par][i]);
  bool flat = false;
  if (kLooks && filter) {
    int share = 0;
#pragma unroll
    for (int i = 0; i < kSampWaves; ++i) share += sh.red[par][i] > m - kNoMass ? sh.share[i] : 0;
    flat = 2 * share > kSampThreads * rounds;
  }
  par ^= 1;
  const bool finite = m > -INFINITY && m < INFINITY;  // and no NaN in the row
  const bool by_bins = filter && finite && !flat;
  if (!finite) {  // the largest number among NaN and infinite logits, 0 where that is infinite
    m = -INFINITY;
#pragma unroll
    for (int k = 0; k < K; ++k) {
      if (k >= rounds) break;
#pragma unroll
      for (int j = 0; j < N; ++j) m = fmaxf(m, e[k][j]);
    }
    m = group_max<64>(m);
    if (lane == 0) sh.red[par][w] = m;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kSampWaves; ++i) m = fmaxf(m, sh.red[par][i]);
    par ^= 1;
    if (!(m > -INFINITY && m < INFINITY)) m = 0.f;
  }
#pragma unroll
  for (int k = 0; k < K; ++k) {
    if (k >= rounds) break;
#pragma unroll
    for (int j = 0; j < N; ++j) e[k][j] = expf(e[k][j] - m);
    if (!by_bins) continue;
    // the most likely token has e == 1, every e is in [0, 1]
    // where all lanes hold the same value, one of them adds for all (rows of 16-bit logits like that are bisected)
    const float e0 = e[k][0];
    const bool same =
        !kLooks && __builtin_amdgcn_ballot_w64(e0 != __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(
                                                                __builtin_bit_cast(int, e0)))) == 0;
    if (same) {
#pragma unroll
      for (int j = 0; j < N; ++j) {
        const uint32_t v = __builtin_bit_cast(uint32_t, e[k][j]);
        const bool all = __builtin_amdgcn_ballot_w64(v != (uint32_t)__builtin_amdgcn_readfirstlane((int)v)) == 0;
        if (v >= kHistLeast && (!all || lane == 0))
          atomicAdd(hist_slot(hist.coarse, v), hist_entry(v) << (all ? 6 : 0));
      }
    } else {
#pragma unroll
      for (int j = 0; j < N; ++j) {
        // a token of no mass adds to one of the bins nobody reads, each lane to its own: no branch
        const float x = e[k][j];
        const uint32_t v = max(__builtin_bit_cast(uint32_t, x), (uint32_t)(kHistBins + lane) << kHistShift);
        atomicAdd(hist_slot(hist.coarse, v), hist_entry(v));
      }
    }
  }

  if (filter) {  // zero the e of every token that does not survive
    float thr;
    int n_equal = INT_MAX, equal = INT_MAX;  // equal: tokens of value thr, or more
    if (by_bins) {
      __syncthreads();
      // the value at which the mass of the values from the top down passes the target
      const u32x4 pair = reinterpret_cast<const u32x4*>(hist.coarse)[kSampThreads - 1 - t];
      mass_t two[2], mine = 0;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int bin = 2 * kHistBins - 1 - (2 * t + i);  // from the top down
        const mass_t entry = ((mass_t)pair[3 - 2 * i] << 32) | pair[2 - 2 * i];
        const mass_t sum = hist_mantissas(entry, bin);
        const int up = mass_shift(bin);
        two[i] = bin < kHistFirst ? 0 : up >= 0 ? sum << up : sum >> -up;
        mine += two[i];
      }
      const mass_t inc = wave_prefix_mass(mine);
      if (lane == kWave - 1) hist.wave_mass[w] = inc;
      __syncthreads();
      static_assert(kSampWaves == 16, "one row of lanes holds the waves' sums");
      const mass_t waves = row_prefix_mass(hist.wave_mass[lane & (kSampWaves - 1)]);  // every row of lanes the same
      const mass_t total = lane_mass(waves, kSampWaves - 1);
      mass_t before = inc - mine + (w > 0 ? lane_mass(waves, w - 1) : 0);
      const mass_t target = (mass_t)((double)fmaxf(p, 0.f) * (double)total);
      if (before <= target && target < before + mine) {  // one lane of the workgroup
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          if (before <= target && target < before + two[i]) {
            const int bin = 2 * kHistBins - 1 - (2 * t + i), up = mass_shift(bin);
            hist.bin = bin;
            hist.goal = up >= 0 ? (target - before) >> up : (target - before) << -up;
          }
          before += two[i];
        }
      }
      __syncthreads();
      uint32_t top = __builtin_amdgcn_readfirstlane(hist.bin);  // the leading bits found so far
#pragma unroll
      for (int k = 0; k < K; ++k) {
        if (k >= rounds) break;
#pragma unroll
        for (int j = 0; j < N; ++j) {
          const uint32_t b = __builtin_bit_cast(uint32_t, e[k][j]);
          if (b >> kHistShift == top) {
            const uint32_t bin = (b >> kHistLast) & ((1 << kHistFine) - 1);
            atomicAdd(&hist.fine[bin], (mass_t)mantissa(b));
            atomicMin(&hist.least[bin], b);
            atomicMax(&hist.most[bin], b);
          }
        }
      }
      __syncthreads();
      if (w == 0) find_in_level<kHistFine>(hist, hist.fine, top, lane, false);
      __syncthreads();
      if (hist.thr == 0) {  // several values in that bin: its last bits
        top = __builtin_amdgcn_readfirstlane(hist.bin);
#pragma unroll
        for (int k = 0; k < K; ++k) {
          if (k >= rounds) break;
#pragma unroll
          for (int j = 0; j < N; ++j) {
            const uint32_t b = __builtin_bit_cast(uint32_t, e[k][j]);
            if (b >> kHistLast == top) atomicAdd(&hist.last[b & ((1 << kHistLast) - 1)], (mass_t)mantissa(b));
          }
        }
        __syncthreads();
        if (w == 0) find_in_level<kHistLast>(hist, hist.last, top, lane, true);
        __syncthreads();
      }
      const uint32_t tb = hist.thr;  // a copy: the cast is applied to a plain scalar
      thr = __builtin_bit_cast(float, tb);
      n_equal = hist.n_equal;
      equal = hist.equal;
    } else {  // NaN or infinite logits, few distinct values: bisection over the element type's patterns
      float z = 0.f, e_lo = INFINITY;
#pragma unroll
      for (int k = 0; k < K; ++k) {
        if (k >= rounds) break;
#pragma unroll
        for (int j = 0; j < N; ++j) {
          z += e[k][j];
          e_lo = fminf(e_lo, e[k][j] > 0.f ? e[k][j] : INFINITY);
        }
      }
      z = block_sum(z);
      const float target = fmaxf(p, 0.f) * z;
      float g_hi = 0.f, e_hi = 1.f;
      // the value looked for is one of the row's, from e_lo to e_hi: two cuts halfway between them, each moving one of
      // them to the nearest value, and a row of one to three values is through (in a row with an infinite maximum the
      // bits alone decide)
      e_lo = finite ? -block_maximum(-e_lo) : 0.f;
      for (int looks = finite ? 2 : 0; looks > 0 && e_lo < e_hi; --looks) {  // the same in every lane
        const float cut = 0.5f * (e_lo + e_hi);
        float g = 0.f, above = INFINITY, up_to = 0.f;
#pragma unroll
        for (int k = 0; k < K; ++k) {
          if (k >= rounds) break;
#pragma unroll
          for (int j = 0; j < N; ++j) {
            const bool over = e[k][j] > cut;
            g += over ? e[k][j] : 0.f;
            above = fminf(above, over ? e[k][j] : INFINITY);
            up_to = fmaxf(up_to, over ? 0.f : e[k][j]);
          }
        }
        g = block_sum(g);
        if (g <= target) {
          g_hi = g;
          e_hi = block_maximum(up_to);
        } else {
          e_lo = -block_maximum(-above);
        }
      }
      thr = e_hi;
      if (!(e_lo >= e_hi)) {
        uint32_t lo = to_key<SH>(-INFINITY), hi = to_key<SH>(m);
        if (e_lo > 0x1p-100f) {
          // between the logits of the two values the looks leave, to within what expf (of a number that is not subnormal),
          // logf and their sums can be off: 2e-7 of every term.  From the type's whole range such rows took 1 to 5 %
          // longer than without the looks.  64 rows of 32,000 fp16 logits, whole range / between: nearly flat about zero,
          // where most patterns lie, 38.3 / 37.6 us, four values 38.7 / 38.0, normal logits cut off above zero 36.4 / 29.7.
          const float a = logf(e_lo), slack = 1e-6f * (1.f + __builtin_fabsf(m) - a);
          lo = max(lo, to_key<SH>(m + a - slack));
          hi = min(hi, to_key<SH>(m + logf(e_hi) + slack) + 1);
        } else {
          g_hi = 0.f;
        }
        while (lo < hi) {  // lo, hi and g are the same in every lane
          const uint32_t mid = lo + ((hi - lo) >> 1);
          const float cut = expf(from_key<SH>(mid) - m);
          float g = 0.f;
#pragma unroll
          for (int k = 0; k < K; ++k) {
            if (k >= rounds) break;
#pragma unroll
            for (int j = 0; j < N; ++j) g += e[k][j] > cut ? e[k][j] : 0.f;
          }
          g = block_sum(g);
          if (g <= target) {
            hi = mid;
            g_hi = g;
          } else {
            lo = mid + 1;
          }
        }
        thr = expf(from_key<SH>(hi) - m);
      }
      if (thr > 0.f) {
        const float r = floorf((target - g_hi) / thr);
        n_equal = r >= 2.0e9f ? INT_MAX : max((int)r + 1, 1);
      }
    }
    if (equal <= n_equal) {  // every token of value thr survives
#pragma unroll
      for (int k = 0; k < K; ++k) {
        if (k >= rounds) break;
#pragma unroll
        for (int j = 0; j < N; ++j) e[k][j] = e[k][j] >= thr ? e[k][j] : 0.f;
      }
    } else {
      // tokens equal to thr survive in id order until n_equal of them have: counted per round and wave, which is the
      // order of the ids, then ranked inside the (round, wave) in which the count passes n_equal
      int cnt[K];
#pragma unroll
      for (int k = 0; k < K; ++k) {
        cnt[k] = 0;
        if (k < rounds) {
#pragma unroll
          for (int j = 0; j < N; ++j) cnt[k] += __builtin_popcountll(__builtin_amdgcn_ballot_w64(e[k][j] == thr));
        }
        if (lane == 0) ired[k * kSampWaves + w] = cnt[k];
      }
      __syncthreads();
      constexpr int kPerWave = kWave / kSampWaves;  // rounds whose counts the lanes of a wave hold at once
      int carry = 0, upto = 0;                      // tokens equal to thr in the rounds before; up to a lane's entry
#pragma unroll
      for (int k = 0; k < K; ++k) {
        if (k % kPerWave == 0) {
          const int at = k * kSampWaves + lane;
          upto = carry + wave_prefix_sum(at < K * kSampWaves ? ired[at] : 0);
          carry = __builtin_amdgcn_readlane(upto, kWave - 1);
        }
        if (k >= rounds) continue;
        const int before = __builtin_amdgcn_readlane(upto, (k % kPerWave) * kSampWaves + w) - cnt[k];
        if (before + cnt[k] <= n_equal) {  // same in every lane of the wave
#pragma unroll
          for (int j = 0; j < N; ++j) e[k][j] = e[k][j] >= thr ? e[k][j] : 0.f;
        } else {
          int rank = before;  // of this lane's first equal token: the equal tokens of the lanes before
#pragma unroll
          for (int j = 0; j < N; ++j) {
            const uint64_t eq = __builtin_amdgcn_ballot_w64(e[k][j] == thr);
            rank = __builtin_amdgcn_mbcnt_hi((uint32_t)(eq >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)eq, rank));
          }
#pragma unroll
          for (int j = 0; j < N; ++j) {
            const float v = e[k][j];
            bool keep = v > thr;
            if (v == thr) keep = rank++ < n_equal;
            e[k][j] = keep ? v : 0.f;
          }
        }
      }
    }
  }

  // the draw: first token, in id order, at which the running sum of e passes uniform * (sum of e)
  float cs[K];
#pragma unroll
  for (int k = 0; k < K; ++k) {
    cs[k] = 0.f;
    if (k >= rounds) continue;
#pragma unroll
    for (int j = 0; j < N; ++j) cs[k] += e[k][j];
    const float v = group_sum<64>(cs[k]);
    if (lane == 0) fred[k][w] = v;
  }
  __syncthreads();
  float round_sum = 0.f;  // lane k: of round k
  if (lane < rounds) {
#pragma unroll
    for (int i = 0; i < kSampWaves; ++i) round_sum += fred[lane][i];
  }
  float tot[K], kept = 0.f;
#pragma unroll
  for (int k = 0; k < K; ++k) {
    tot[k] = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, round_sum), k));
    kept += tot[k];
  }
  const float goal = uniform * kept;
  int kd = K;  // the round in which the running sum passes the goal
  float before_kd = 0.f, run = 0.f;
#pragma unroll
  for (int k = 0; k < K; ++k) {
    if (kd == K && run + tot[k] > goal) {
      kd = k;
      before_kd = run;
    }
    run += tot[k];
  }
  float mine = 0.f;
#pragma unroll
  for (int k = 0; k < K; ++k) mine = k == kd ? cs[k] : mine;
  float finc = mine;
#pragma unroll
  for (int d = 1; d < kWave; d <<= 1) {
    const float up = __shfl_up(finc, d, kWave);
    if (lane >= d) finc += up;
  }
  if (lane == kWave - 1) sh.fpart[w] = finc;
  __syncthreads();
  float running = before_kd;
#pragma unroll
  for (int i = 0; i < kSampWaves - 1; ++i) running += i < w ? sh.fpart[i] : 0.f;
  running += finc - mine;
  int found = INT_MAX;
#pragma unroll
  for (int k = 0; k < K; ++k) {
    if (k != kd) continue;  // same in every lane
#pragma unroll
    for (int j = 0; j < N; ++j) {
      const float v = e[k][j];
      running += v;
      if (v > 0.f && running > goal && found == INT_MAX) found = (t + k * kSampThreads) * N + j;
    }
  }
  if (found != INT_MAX) atomicMin(&sh.found, found);
  __syncthreads();
  if (sh.found == INT_MAX) {  // same in every lane
    // rounding can leave the goal a hair above the sums of the round it was placed in: then the next surviving
    // token, or the last one of the row
    int found_after = INT_MAX, last = -1;
#pragma unroll
    for (int k = 0; k < K; ++k) {
      if (k >= rounds) break;
#pragma unroll
      for (int j = 0; j < N; ++j) {
        const int i = (t + k * kSampThreads) * N + j;
        if (e[k][j] > 0.f) {
          last = i;
          if (k > kd && found_after == INT_MAX) found_after = i;
        }
      }
    }
    if (found_after != INT_MAX) atomicMin(&sh.found_after, found_after);
    if (last >= 0) atomicMax(&sh.last, last);
    __syncthreads();
  }
  if (t == 0) a.out[row] = sh.found != INT_MAX ? sh.found : sh.found_after != INT_MAX ? sh.found_after : max(sh.last, 0);
}

template <typename E>
static int launch_sample(const SampArgs& a, int64_t rows, hipStream_t st) {
  dim3 grid((unsigned)rows), block(kSampThreads);
  const bool rows_aligned = aligned16(a.logits) && (a.row_stride * Logit<E>::kBytes) % 16 == 0;
  if (rows_aligned && a.V <= kSampThreads * kSampShortFloats) {
    hipLaunchKernelGGL((sample_rows_kernel<E, kSampShortFloats>), grid, block, 0, st, a);
  } else if (rows_aligned && a.V <= kSampThreads * kSampRegFloats) {
    hipLaunchKernelGGL((sample_rows_kernel<E, kSampRegFloats>), grid, block, 0, st, a);
  } else if (a.V <= kSampLdsFloats) {
    const size_t lds = (size_t)a.V * sizeof(float);
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&sample_top_p_kernel<E, true>),
                              hipFuncAttributeMaxDynamicSharedMemorySize, kSampLdsFloats * (int)sizeof(float));
    hipLaunchKernelGGL((sample_top_p_kernel<E, true>), grid, block, lds, st, a);
  } else {
    hipLaunchKernelGGL((sample_top_p_kernel<E, false>), grid, block, 0, st, a);
  }
  return launch_status();
}

}  // namespace ph

using namespace ph;

extern "C" int ph_sample_top_p(const void* logits, int64_t row_stride, const float* temperature, const float* top_p,
                               const float* uniform, int64_t* out_ids, int64_t rows, int64_t vocab, int dtype,
                               void* stream) {
  if (rows < 0 || vocab <= 0 || vocab >= ((int64_t)1 << 30) || row_stride < vocab) return PH_ERR_ARG;
  if (dtype != PH_F16 && dtype != PH_BF16 && dtype != PH_F32) return PH_ERR_DTYPE;
  if (rows == 0) return PH_OK;
  if (!logits || !uniform || !out_ids) return PH_ERR_ARG;
  if (rows > 0x7fffffff) return PH_ERR_ARG;
  const SampArgs a{logits, row_stride, temperature, top_p, uniform, out_ids, (int)vocab, nullptr, 0};
  hipStream_t st = (hipStream_t)stream;
  if (dtype == PH_F16) return launch_sample<F16>(a, rows, st);
  if (dtype == PH_BF16) return launch_sample<BF16>(a, rows, st);
  return launch_sample<F32>(a, rows, st);
}

template <typename E>
static int launch_probs(const SampArgs& a, int64_t rows, hipStream_t st) {
  dim3 grid((unsigned)rows), block(kSampThreads);
  if (a.V <= kSampLdsFloats) {
    const size_t lds = (size_t)a.V * sizeof(float);
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&sample_top_p_kernel<E, true>),
                              hipFuncAttributeMaxDynamicSharedMemorySize, kSampLdsFloats * (int)sizeof(float));
    hipLaunchKernelGGL((sample_top_p_kernel<E, true>), grid, block, lds, st, a);
  } else {
    hipLaunchKernelGGL((sample_top_p_kernel<E, false>), grid, block, 0, st, a);
  }
  return launch_status();
}

extern "C" int ph_top_p_probs(const void* logits, int64_t row_stride, const float* temperature, const float* top_p,
                              float* probs, int64_t probs_stride, int64_t rows, int64_t vocab, int dtype,
                              void* stream) {
  if (rows < 0 || vocab <= 0 || vocab >= ((int64_t)1 << 30) || row_stride < vocab || probs_stride < vocab)
    return PH_ERR_ARG;
  if (dtype != PH_F16 && dtype != PH_BF16 && dtype != PH_F32) return PH_ERR_DTYPE;
  if (rows == 0) return PH_OK;
  if (!logits || !probs || rows > 0x7fffffff) return PH_ERR_ARG;
  const SampArgs a{logits, row_stride, temperature, top_p, nullptr, nullptr, (int)vocab, probs, probs_stride};
  hipStream_t st = (hipStream_t)stream;
  if (dtype == PH_F16) return launch_probs<F16>(a, rows, st);
  if (dtype == PH_BF16) return launch_probs<BF16>(a, rows, st);
  return launch_probs<F32>(a, rows, st);
}
