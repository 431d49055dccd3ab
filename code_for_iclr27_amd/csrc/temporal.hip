// Op-level temporal scoring kernels with the reference's per-op contracts:
//   temporal_probabilities  csrc/scoring.cu:32-66   (masked, scaled, dtype-rounded softmax)
//   temporal_risk           csrc/scoring.cu:68-128  (min/max margin drop -> Bernoulli risk)
//   pool                    csrc/scoring.cu:190-203 (segmented sliding max)
//   decision_risk_scores    csrc/cache_legacy.cu:63-135 (legacy single-query scorer)
// Arithmetic follows the reference operation by operation (the library is built with
// -ffp-contract=off so no multiply-add is fused); reductions are wave64-native (butterfly
// within a wave, LDS across waves), so sums may differ from the reference's 256-lane tree in
// the last bits.

#include <algorithm>
#include <cmath>

#include "lr_common.hpp"

namespace lr {
namespace {

template <bool kMax>
__device__ __forceinline__ float wave_reduce(float v) {
#pragma unroll
  for (int offset = 32; offset > 0; offset >>= 1) {
    const float o = __shfl_xor(v, offset, 64);
    v = kMax ? fmaxf(v, o) : v + o;
  }
  return v;
}

// Block-wide reduction over WAVES waves; every thread receives the result. `scratch` holds one
// value a wave and is used once (no barrier before its reuse).
template <bool kMax, int WAVES>
__device__ __forceinline__ float block_reduce(float v, float* scratch) {
  v = wave_reduce<kMax>(v);
  const int wave = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) scratch[wave] = v;
  __syncthreads();
  float r = scratch[0];
#pragma unroll
  for (int w = 1; w < WAVES; ++w) r = kMax ? fmaxf(r, scratch[w]) : r + scratch[w];
  return r;
}

template <typename T>
__device__ __forceinline__ float round_to(float x);
template <>
__device__ __forceinline__ float round_to<float>(float x) { return x; }
template <>
__device__ __forceinline__ float round_to<_Float16>(float x) { return static_cast<float>(static_cast<_Float16>(x)); }
template <>
__device__ __forceinline__ float round_to<__bf16>(float x) {
  return static_cast<float>(static_cast<__bf16>(x));
}

template <typename T>
__device__ __forceinline__ float load_as_float(const T* p, int64_t i);
template <>
__device__ __forceinline__ float load_as_float<float>(const float* p, int64_t i) { return p[i]; }
template <>
__device__ __forceinline__ float load_as_float<double>(const double* p, int64_t i) {
  return static_cast<float>(p[i]);
}
template <>
__device__ __forceinline__ float load_as_float<_Float16>(const _Float16* p, int64_t i) {
  return static_cast<float>(p[i]);
}
template <>
__device__ __forceinline__ float load_as_float<__bf16>(const __bf16* p, int64_t i) {
  return static_cast<float>(p[i]);
}

// One block per (query, group) row. Thread t owns positions t, t + THREADS, ...: CACHE of them in
// registers (the masked logits, then the exponentials), so a row is read once. A row is short work
// (a 8B head: 9 positions a thread), so its time is its chain of memory and barrier latencies:
// every load of the row, the projected values included, is issued before the first is used
// (clamped to the row; a load under the bounds check would be waited for inside it). Measured (64
// queries x 4 groups, calls back to back, us, against 256 threads a row and loads in bounded
// loops): 2,250 keys 4.7 against 6.3, 16,000 10.8 against 41.6, 33,792 30 against 94.
// CACHE = 0: longer rows, the masked logits read again in each of the three phases.
template <typename T, int THREADS, int CACHE>
__global__ __launch_bounds__(THREADS) void probabilities_kernel(
    const T* __restrict__ logits, const float* __restrict__ projected,
    const int64_t* __restrict__ query_positions, const float* __restrict__ key_positions,
    float* __restrict__ probabilities, float* __restrict__ output_projection, int64_t groups,
    int64_t length, float scale) {
  constexpr int WAVES = THREADS / 64;
  __shared__ float scratch[3][WAVES];
  const int64_t row = blockIdx.x;
  const int64_t group = row % groups;
  const int64_t query = row / groups;
  const float query_position = static_cast<float>(query_positions[query]);
  const T* in = logits + row * length;
  float* out = probabilities + row * length;
  const float* pv = projected + group * length;
  const int64_t first = threadIdx.x;
  // Reference compares float key positions against the int64 query position promoted
  // to float (csrc/scoring.cu:46).
  auto masked = [&](float logit, float key_position) -> float {
    const float rounded = round_to<T>(logit * scale);
    return key_position <= query_position ? rounded : -INFINITY;
  };
  float maximum = -INFINITY, denominator = 0.0f, projection = 0.0f;
  if constexpr (CACHE > 0) {
    float x[CACHE], k[CACHE], v[CACHE];
#pragma unroll
    for (int i = 0; i < CACHE; ++i) {
      const int64_t at = first + i * THREADS < length ? first + i * THREADS : length - 1;
      x[i] = load_as_float<T>(in, at);
      k[i] = key_positions[at];
      v[i] = pv[at];
    }
#pragma unroll
    for (int i = 0; i < CACHE; ++i) {
      x[i] = first + i * THREADS < length ? masked(x[i], k[i]) : -INFINITY;
      maximum = fmaxf(maximum, x[i]);
    }
    maximum = block_reduce<true, WAVES>(maximum, scratch[0]);
#pragma unroll
    for (int i = 0; i < CACHE; ++i) {
      if (first + i * THREADS >= length) break;
      x[i] = expf(x[i] - maximum);
      denominator += x[i];
    }
    denominator = block_reduce<false, WAVES>(denominator, scratch[1]);
#pragma unroll
    for (int i = 0; i < CACHE; ++i) {
      if (first + i * THREADS >= length) break;
      const float p = x[i] / denominator;
      out[first + i * THREADS] = p;
      projection += p * v[i];
    }
  } else {
    constexpr int U = 8;  // positions whose loads are in flight together
    auto visit = [&](auto&& use) {
      for (int64_t base = first; base < length; base += U * THREADS) {
        float x[U], k[U], v[U];
#pragma unroll
        for (int i = 0; i < U; ++i) {
          const int64_t at = base + i * THREADS < length ? base + i * THREADS : length - 1;
          x[i] = load_as_float<T>(in, at);
          k[i] = key_positions[at];
          v[i] = pv[at];
        }
#pragma unroll
        for (int i = 0; i < U; ++i)
          if (base + i * THREADS < length) use(base + i * THREADS, masked(x[i], k[i]), v[i]);
      }
    };
    visit([&](int64_t, float z, float) { maximum = fmaxf(maximum, z); });
    maximum = block_reduce<true, WAVES>(maximum, scratch[0]);
    visit([&](int64_t, float z, float) { denominator += expf(z - maximum); });
    denominator = block_reduce<false, WAVES>(denominator, scratch[1]);
    visit([&](int64_t at, float z, float value) {
      const float p = expf(z - maximum) / denominator;
      out[at] = p;
      projection += p * value;
    });
  }
  projection = block_reduce<false, WAVES>(projection, scratch[2]);
  if (threadIdx.x == 0) output_projection[row] = projection;
}

__device__ __forceinline__ double softplus64(double v) { return v > 20.0 ? v : log1p(exp(v)); }

__device__ __forceinline__ double risk64(double margin, double probability, double base_softplus,
                                         float drop) {
  const double compared = margin - static_cast<double>(drop);
  return fmax(0.0, probability * (margin - compared) - base_softplus + softplus64(compared));
}

// A block of 16 waves takes 64 candidates (one a lane); wave w visits queries w, w + 16, ..., four
// at a time with every group's probability loaded before the first is used. The margin drop of one
// (query, candidate) sums the groups in order g = 0..G-1 exactly like the reference. Any
// non-finite drop makes the candidate's score NaN. There are only as many blocks as 64-candidate
// columns (35 for an 8B head), so the depth of a wave's loads sets the time: 16 waves of four
// queries take 5.4 us for 64 queries x 4 groups x 2,218 candidates, four waves one query at a time
// took 14.5 (calls back to back).
constexpr int kRiskCandidates = 64;
constexpr int kRiskWaves = 16, kFewRiskWaves = 4;
constexpr int kRiskQueries = 4;

// GROUPS: the group count known at compile time (loads of all groups in flight), or 0.
template <int GROUPS, int WAVES>
__global__ __launch_bounds__(kRiskCandidates* WAVES) void risk_kernel(
    const float* __restrict__ probabilities, const float* __restrict__ output_projection,
    const float* __restrict__ projected, const float* __restrict__ margin,
    float* __restrict__ result, int64_t window, int64_t groups_in, int64_t length, int64_t first,
    int64_t count, float epsilon, int accumulate) {
  __shared__ float minimums[WAVES][kRiskCandidates];
  __shared__ float maximums[WAVES][kRiskCandidates];
  __shared__ int bad[WAVES][kRiskCandidates];
  __shared__ double terms[2];
  __shared__ double upper_risk[kRiskCandidates];
  const int64_t groups = GROUPS ? GROUPS : groups_in;
  const int lane = threadIdx.x % kRiskCandidates;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kRiskCandidates);
  const int64_t candidate = static_cast<int64_t>(blockIdx.x) * kRiskCandidates + lane;
  const bool live = candidate < count;
  const int64_t position = first + (live ? candidate : count - 1);
  float minimum = INFINITY, maximum = -INFINITY;
  int nonfinite = 0;
  auto drop_term = [&](float p, float value, float output) {
    const float ratio = p / fmaxf(1.0f - p, epsilon);
    return ratio * (value - output);
  };
  auto visit = [&](float drop) {
    if (!isfinite(drop)) nonfinite = 1;
    minimum = fminf(minimum, drop);
    maximum = fmaxf(maximum, drop);
  };
  if constexpr (GROUPS > 0) {
    float value[GROUPS];
#pragma unroll
    for (int g = 0; g < GROUPS; ++g) value[g] = projected[g * length + position];
    for (int64_t q0 = wave; q0 < window; q0 += WAVES * kRiskQueries) {
      float p[kRiskQueries][GROUPS];
#pragma unroll
      for (int j = 0; j < kRiskQueries; ++j) {
        const int64_t q = q0 + j * WAVES < window ? q0 + j * WAVES : q0;
#pragma unroll
        for (int g = 0; g < GROUPS; ++g) p[j][g] = probabilities[(q * GROUPS + g) * length + position];
      }
#pragma unroll
      for (int j = 0; j < kRiskQueries; ++j) {
        const int64_t q = q0 + j * WAVES;
        if (q >= window) break;
        float drop = 0.0f;
#pragma unroll
        for (int g = 0; g < GROUPS; ++g)
          drop += drop_term(p[j][g], value[g], output_projection[q * GROUPS + g]);
        visit(drop);
      }
    }
  } else {
    for (int64_t q = wave; q < window; q += WAVES) {
      float drop = 0.0f;
      for (int64_t g = 0; g < groups; ++g)
        drop += drop_term(probabilities[(q * groups + g) * length + position],
                          projected[g * length + position], output_projection[q * groups + g]);
      visit(drop);
    }
  }
  minimums[wave][lane] = minimum;
  maximums[wave][lane] = maximum;
  bad[wave][lane] = nonfinite;
  const double m = static_cast<double>(margin[0]);
  if (threadIdx.x == kRiskCandidates * (WAVES - 1)) {  // the margin's terms, once
    terms[0] = 1.0 / (1.0 + exp(-m));
    terms[1] = softplus64(m);
  }
  __syncthreads();
  // Wave 0 takes the risk of the minimum, wave 1 that of the maximum.
  double risk = 0.0;
  if (wave < 2) {
    for (int w = 0; w < WAVES; ++w) {
      minimum = fminf(minimum, minimums[w][lane]);
      maximum = fmaxf(maximum, maximums[w][lane]);
      nonfinite |= bad[w][lane];
    }
    risk = risk64(m, terms[0], terms[1], wave ? maximum : minimum);
    if (wave) upper_risk[lane] = risk;
  }
  __syncthreads();
  if (wave == 0 && live) {
    float score = nonfinite ? NAN : static_cast<float>(fmax(risk, upper_risk[lane]));
    if (accumulate) score = __builtin_elementwise_maximum(score, result[candidate]);
    result[candidate] = score;
  }
}

// Sliding max of odd width inside each segment; NaN neighbours are ignored as by fmaxf and
// out-of-segment neighbours do not exist (csrc/scoring.cu:190-203). Block tile + halo in LDS.
// Workgroup (0, 0) also zeroes `clear[0, clear_words)` when given (the selection's counters, so
// that a following selection needs no launch of its own to reset them).
constexpr int kPoolThreads = 256;

__global__ __launch_bounds__(kPoolThreads) void pool_kernel(const float* __restrict__ scores,
                                                             int64_t total,
                                                             const int64_t* __restrict__ bounds,
                                                             float* __restrict__ output,
                                                             int half, int use_lds,
                                                             uint32_t* __restrict__ clear,
                                                             int clear_words) {
  extern __shared__ float tile[];
  if (clear != nullptr && blockIdx.x == 0 && blockIdx.y == 0)
    for (int i = threadIdx.x; i < clear_words; i += kPoolThreads) clear[i] = 0;
  const int64_t segment = blockIdx.y;
  int64_t begin = bounds[segment], end = bounds[segment + 1];
  if (begin < 0) begin = 0;
  if (end > total) end = total;
  const int64_t tile_start = begin + static_cast<int64_t>(blockIdx.x) * kPoolThreads;
  if (tile_start >= end) return;
  const int64_t position = tile_start + threadIdx.x;
  if (use_lds) {
    const int span = kPoolThreads + 2 * half;
    for (int i = threadIdx.x; i < span; i += kPoolThreads) {
      const int64_t p = tile_start - half + i;
      tile[i] = (p >= begin && p < end) ? scores[p] : -INFINITY;
    }
    __syncthreads();
    if (position >= end) return;
    float value = -INFINITY;
    for (int o = 0; o <= 2 * half; ++o) value = fmaxf(value, tile[threadIdx.x + o]);
    output[position] = value;
  } else {
    if (position >= end) return;
    float value = -INFINITY;
    for (int64_t o = -half; o <= half; ++o) {
      const int64_t n = position + o;
      if (n >= begin && n < end) value = fmaxf(value, scores[n]);
    }
    output[position] = value;
  }
}

__device__ __forceinline__ double stable_sigmoid(double v) {
  if (v >= 0.0) return 1.0 / (1.0 + exp(-v));
  const double e = exp(v);
  return e / (1.0 + e);
}

__device__ __forceinline__ double stable_softplus(double v) {
  if (v > 20.0) return v + log1p(exp(-v));
  return log1p(exp(v));
}

// One 256-thread block per candidate. The margin drop is a long mixed-sign sum whose
// cancellation amplifies any change of summation order, so this legacy op keeps the
// reference's order (csrc/cache_legacy.cu:98-121): thread t accumulates terms t, t+256, ...,
// then an LDS tree halves the 256 partials.
template <typename T>
__global__ __launch_bounds__(256) void decision_risk_kernel(
    float* __restrict__ scores, const float* __restrict__ probabilities,
    const T* __restrict__ values, const float* __restrict__ head_outputs,
    const float* __restrict__ gradients, int64_t groups, int64_t candidates, int64_t head_dim,
    double base_margin, float epsilon) {
  __shared__ float reduction[256];
  const int64_t candidate = blockIdx.x;
  float partial = 0.0f;
  const int64_t terms = groups * head_dim;
  for (int64_t index = threadIdx.x; index < terms; index += 256) {
    const int64_t group = index / head_dim;
    const int64_t d = index % head_dim;
    const float alpha = probabilities[group * candidates + candidate];
    const float denominator = fmaxf(1.0f - alpha, epsilon);
    const float value = load_as_float<T>(values, candidate * head_dim + d);
    const float local_delta = alpha / denominator * (value - head_outputs[group * head_dim + d]);
    partial += gradients[group * head_dim + d] * local_delta;
  }
  reduction[threadIdx.x] = partial;
  __syncthreads();
  for (int stride = 128; stride > 0; stride >>= 1) {
    if (threadIdx.x < stride) reduction[threadIdx.x] += reduction[threadIdx.x + stride];
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    const double compared = base_margin - static_cast<double>(reduction[0]);
    const double probability = stable_sigmoid(base_margin);
    double kl = probability * (base_margin - compared) - stable_softplus(base_margin) +
                stable_softplus(compared);
    if (kl < 0.0) kl = 0.0;
    scores[candidate] = static_cast<float>(kl);
  }
}

constexpr int64_t kLaunchThreads = int64_t{1} << 32;

template <typename T>
int launch_probabilities(const void* logits, const float* projected, const int64_t* qpos,
                         const float* kpos, int64_t window, int64_t groups, int64_t length,
                         float scale, float* probabilities, float* output_projection,
                         hipStream_t stream) {
  const int64_t rows = window * groups;
  const T* in = static_cast<const T*>(logits);
  auto launch = [&](auto kernel, int threads) {
    kernel<<<static_cast<unsigned>(rows), threads, 0, stream>>>(
        in, projected, qpos, kpos, probabilities, output_projection, groups, length, scale);
  };
  // The smallest cache that holds the row: unused positions cost loads of the row's last one.
  if (length <= 256 * 4) launch(probabilities_kernel<T, 256, 4>, 256);
  else if (length <= 256 * 9) launch(probabilities_kernel<T, 256, 9>, 256);
  else if (length <= 256 * 16) launch(probabilities_kernel<T, 256, 16>, 256);
  // a launch has fewer than 2^32 threads: past 2^22 rows the blocks stay narrow
  else if (rows >= kLaunchThreads / 1024) launch(probabilities_kernel<T, 256, 0>, 256);
  else if (length <= 1024 * 16) launch(probabilities_kernel<T, 1024, 16>, 1024);
  else launch(probabilities_kernel<T, 1024, 0>, 1024);
  return check_launch("temporal_probabilities");
}

}  // namespace
}  // namespace lr

using namespace lr;

extern "C" int lr_temporal_probabilities(const void* logits, int logits_dtype,
                                         const float* projected, const int64_t* query_positions,
                                         const float* key_positions, int64_t window,
                                         int64_t groups, int64_t length, float scale,
                                         float* probabilities, float* output_projection,
                                         void* stream) {
  clear_error();
  LR_REQUIRE(logits_dtype == LR_DTYPE_F32 || logits_dtype == LR_DTYPE_F16 ||
                 logits_dtype == LR_DTYPE_BF16,
             "Only FP32/FP16/BF16 scores are supported");
  LR_REQUIRE(window > 0 && groups > 0 && length > 0, "Empty attention dimensions");
  LR_REQUIRE(window * groups <= 2147483647LL, "Empty attention dimensions");
  LR_REQUIRE(logits && projected && query_positions && key_positions && probabilities &&
                 output_projection,
             "Expected contiguous CUDA tensor");
  const hipStream_t s = as_stream(stream);
  switch (logits_dtype) {
    case LR_DTYPE_F32:
      return launch_probabilities<float>(logits, projected, query_positions, key_positions, window,
                                         groups, length, scale, probabilities, output_projection, s);
    case LR_DTYPE_F16:
      return launch_probabilities<_Float16>(logits, projected, query_positions, key_positions, window,
                                          groups, length, scale, probabilities, output_projection, s);
    default:
      return launch_probabilities<__bf16>(logits, projected, query_positions, key_positions,
                                                   window, groups, length, scale, probabilities,
                                                   output_projection, s);
  }
}

namespace lr {
namespace {

int risk_scores(const float* probabilities, const float* output_projection, const float* projected,
                const float* margin, int64_t window, int64_t groups, int64_t length, int64_t first,
                int64_t last, double epsilon, float* result, int accumulate, void* stream) {
  LR_REQUIRE(window > 0 && groups > 0 && first >= 0 && last > first && last <= length &&
                 epsilon > 0,
             "Invalid risk interval");
  LR_REQUIRE(probabilities && output_projection && projected && margin && result,
             "Expected contiguous CUDA tensor");
  const int64_t count = last - first;
  const hipStream_t s = as_stream(stream);
  const float eps = static_cast<float>(epsilon);
  // As many candidates a launch as its threads (fewer than 2^32) allow.
  constexpr int64_t kMost = (kLaunchThreads / (kRiskCandidates * kRiskWaves) - 1) * kRiskCandidates;
  // Few queries leave most of sixteen waves without one: four (8 queries, one group, 60,000 candidates
  // 4.2 us against 5.5).
  const bool few = window <= 2 * kFewRiskWaves;
  auto launch = [&](auto many_kernel, auto few_kernel) {
    for (int64_t done = 0; done < count; done += kMost) {
      const int64_t here = std::min(kMost, count - done);
      const dim3 grid(static_cast<unsigned>(ceil_div(here, kRiskCandidates)));
      (few ? few_kernel : many_kernel)<<<grid, kRiskCandidates * (few ? kFewRiskWaves : kRiskWaves), 0, s>>>(
          probabilities, output_projection, projected, margin, result + done, window, groups,
          length, first + done, here, eps, accumulate);
    }
  };
  switch (groups) {
    case 1: launch(risk_kernel<1, kRiskWaves>, risk_kernel<1, kFewRiskWaves>); break;
    case 2: launch(risk_kernel<2, kRiskWaves>, risk_kernel<2, kFewRiskWaves>); break;
    case 4: launch(risk_kernel<4, kRiskWaves>, risk_kernel<4, kFewRiskWaves>); break;
    case 6: launch(risk_kernel<6, kRiskWaves>, risk_kernel<6, kFewRiskWaves>); break;
    case 8: launch(risk_kernel<8, kRiskWaves>, risk_kernel<8, kFewRiskWaves>); break;
    default: launch(risk_kernel<0, kRiskWaves>, risk_kernel<0, kFewRiskWaves>); break;
  }
  return check_launch("temporal_risk");
}

}  // namespace
}  // namespace lr

extern "C" int lr_temporal_risk(const float* probabilities, const float* output_projection,
                                const float* projected, const float* margin, int64_t window,
                                int64_t groups, int64_t length, int64_t first, int64_t last,
                                double epsilon, float* result, void* stream) {
  clear_error();
  return risk_scores(probabilities, output_projection, projected, margin, window, groups, length,
                     first, last, epsilon, result, 0, stream);
}

extern "C" int lr_temporal_risk_max(const float* probabilities, const float* output_projection,
                                    const float* projected, const float* margin, int64_t window,
                                    int64_t groups, int64_t length, int64_t first, int64_t last,
                                    double epsilon, float* result, void* stream) {
  clear_error();
  return risk_scores(probabilities, output_projection, projected, margin, window, groups, length,
                     first, last, epsilon, result, 1, stream);
}

namespace lr {

int launch_pool(const float* scores, int64_t total, const int64_t* bounds, int64_t segments,
                int64_t max_count, int64_t width, float* out, uint32_t* clear, int clear_words,
                hipStream_t stream) {
  const int half = static_cast<int>(width / 2);
  const int use_lds = width <= 4097 ? 1 : 0;
  const size_t lds = use_lds ? (kPoolThreads + 2 * half) * sizeof(float) : 0;
  dim3 grid(static_cast<unsigned>(ceil_div(max_count, kPoolThreads)),
            static_cast<unsigned>(segments));
  pool_kernel<<<grid, kPoolThreads, lds, stream>>>(scores, total, bounds, out, half, use_lds,
                                                   clear, clear_words);
  return check_launch("pool");
}

}  // namespace lr

extern "C" int lr_pool(const float* scores, int64_t total, const int64_t* bounds,
                       int64_t segments, int64_t max_count, int64_t width, float* out,
                       void* stream) {
  clear_error();
  LR_REQUIRE(segments >= 1 && total >= 0, "Invalid pool layout");
  LR_REQUIRE(width > 0 && width % 2 == 1 && max_count > 0, "Invalid pool configuration");
  LR_REQUIRE(segments <= 65535, "Invalid pool layout");
  if (total == 0) return LR_OK;
  LR_REQUIRE(scores && bounds && out, "Expected contiguous CUDA tensor");
  return launch_pool(scores, total, bounds, segments, max_count, width, out, nullptr, 0,
                     as_stream(stream));
}

extern "C" int lr_decision_risk_scores(const float* probabilities, const void* values,
                                       int values_dtype, const float* head_outputs,
                                       const float* gradients, int64_t groups,
                                       int64_t candidates, int64_t head_dim, double base_margin,
                                       double epsilon, float* scores, void* stream) {
  clear_error();
  LR_REQUIRE(epsilon > 0.0 && epsilon < 1.0, "denominator_epsilon must be in (0,1)");
  LR_REQUIRE(groups >= 0 && candidates >= 0 && head_dim >= 0, "candidate count mismatch");
  LR_REQUIRE(values_dtype >= LR_DTYPE_F32 && values_dtype <= LR_DTYPE_BF16, "Invalid dtype");
  if (candidates == 0) return LR_OK;
  LR_REQUIRE(probabilities && values && head_outputs && gradients && scores,
             "probabilities must be CUDA");
  LR_REQUIRE(candidates <= 2147483647LL, "candidate count mismatch");
  const int64_t blocks = candidates;
  const hipStream_t s = as_stream(stream);
  const float eps = static_cast<float>(epsilon);
  switch (values_dtype) {
    case LR_DTYPE_F32:
      decision_risk_kernel<float><<<blocks, 256, 0, s>>>(
          scores, probabilities, static_cast<const float*>(values), head_outputs, gradients, groups,
          candidates, head_dim, base_margin, eps);
      break;
    case LR_DTYPE_F64:
      decision_risk_kernel<double><<<blocks, 256, 0, s>>>(
          scores, probabilities, static_cast<const double*>(values), head_outputs, gradients,
          groups, candidates, head_dim, base_margin, eps);
      break;
    case LR_DTYPE_F16:
      decision_risk_kernel<_Float16><<<blocks, 256, 0, s>>>(
          scores, probabilities, static_cast<const _Float16*>(values), head_outputs, gradients,
          groups, candidates, head_dim, base_margin, eps);
      break;
    default:
      decision_risk_kernel<__bf16><<<blocks, 256, 0, s>>>(
          scores, probabilities, static_cast<const __bf16*>(values), head_outputs,
          gradients, groups, candidates, head_dim, base_margin, eps);
      break;
  }
  return check_launch("decision_risk_scores");
}
