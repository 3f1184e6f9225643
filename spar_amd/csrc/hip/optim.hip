// Optimizer-side kernels: the AdamW update, the scaled sum-of-squares summary
// behind the global gradient norm, and in-place gradient scaling.
//
// Replaces kernels K16-K18 of src/backend/cuda_kernels.cu (gradient_norm_kernel
// :390-424, scale_in_place_kernel :426-433, adamw_kernel :435-455) behind the
// same entry points (cuda_kernels.hpp:118-128).  All three are HBM-bound
// streams; the arithmetic is IEEE double exactly as the reference's CPU loops
// write it (optim/adamw.cpp:50-60, training/gradients.cpp:107-111), so the
// updated values are the CPU path's bits.
//
// Design for CDNA4:
//  * AdamW and scaling read and write 16-byte vectors per lane in tiles of
//    consecutive vectors, the layout of the elementwise kernels.  AdamW
//    moves 28 bytes per fp32 element (four reads, three writes) and spends
//    about 70 fp64 operations on it (two IEEE divides, one correctly rounded
//    square root): on MI355X that is under half of the fp64 rate at the HBM
//    bound, so the update stays memory-bound without approximating a divide.
//  * The norm summary reads the gradient once across the whole chip (the
//    reference runs one 256-thread block).  Each lane keeps a power-of-two
//    scaled sum of squares: for fp32 input every square is exact in double
//    and no sum of them can overflow, so the scale exponent stays 0; for fp64
//    input the exponent tracks the largest element so far and rescaling is an
//    exact ldexp rather than the reference's division per element.  A lane
//    whose sum turns out non-finite saw an infinity or NaN and re-reads its
//    own elements with the reference's per-element classification, so the
//    common case carries no per-element flag work.  Block partials are
//    combined in a fixed order by one block, so the result is deterministic.
#include <hip/hip_runtime.h>

#include <math.h>

#include "common.hpp"

namespace spar_hip {
namespace {

constexpr int kThreads = 256;
// Streaming kernels use single-wave workgroups (see elementwise.hip).
constexpr int kVectorThreads = 64;
constexpr uint64_t kMaxGrid = uint64_t{1} << 20;

uint32_t scalar_grid(uint64_t count, const DeviceGuard& guard) {
  uint64_t blocks = (count + kThreads - 1) / kThreads;
  const uint64_t cap = static_cast<uint64_t>(guard.multiprocessors) * 16;
  if (blocks > cap) blocks = cap;
  if (blocks == 0) blocks = 1;
  return static_cast<uint32_t>(blocks);
}

// ------------------------------------------------------------------ AdamW

// Per-launch constants of one AdamW step.  `one_minus_beta*` and
// `decay_factor` (1 - lr * weight_decay) are the values the reference forms
// per element and per call; forming them once gives the same doubles.
struct AdamwStep {
  double learning_rate;
  double beta1;
  double beta2;
  double epsilon;
  double first_correction;
  double second_correction;
  double one_minus_beta1;
  double one_minus_beta2;
  double decay_factor;
};

// optim/adamw.cpp:50-60 for one element.  The moments are rounded to T when
// stored and read back before the bias correction, as the reference's loop
// does; every operation is a separately rounded IEEE double operation (the
// library is compiled without contraction).
template <typename T>
__device__ __forceinline__ void adamw_element(T& parameter, T gradient, T& first, T& second,
                                              const AdamwStep& s) {
  const double g = static_cast<double>(gradient);
  first = static_cast<T>(s.beta1 * static_cast<double>(first) + s.one_minus_beta1 * g);
  second = static_cast<T>(s.beta2 * static_cast<double>(second) + s.one_minus_beta2 * g * g);
  const double corrected_first = static_cast<double>(first) / s.first_correction;
  const double corrected_second = static_cast<double>(second) / s.second_correction;
  const double decayed = static_cast<double>(parameter) * s.decay_factor;
  parameter = static_cast<T>(decayed - s.learning_rate * corrected_first /
                                           (sqrt(corrected_second) + s.epsilon));
}

// Many tensors in one launch.  A model's parameter list is mostly small
// tensors: GPT-2 small's 148 took 592 launches a step (partial, combine,
// scale and AdamW for each), whose boundaries and host time came to 2.9 ms
// for 4 GB moved.  A launch takes up to N of them: their work is numbered in
// units (tiles or segments, each tensor's consecutive), and a wave finds the
// tensor of a unit by comparing the units' starts, one lane per tensor (a
// vector load and a ballot per 64 tensors).  N is what keeps the kernel
// arguments under 4 KiB.  N = 1 has nothing to look up and is also the form
// of a tensor of kOwnLaunchBytes or more: it fills the chip by itself, and
// without the lookup's latency ahead of every wave's loads 124M float32
// elements scale in 149 us instead of 155.
template <int N>
struct UnitMap {
  uint32_t tensors = 0;
  uint32_t units = 0;
  uint32_t first[N];  // first unit of each tensor, increasing

  __host__ bool accepts(uint64_t more) const {
    return tensors < static_cast<uint32_t>(N) && units + more <= kIndex32Limit;
  }
  __host__ void append(uint64_t more) {
    first[tensors++] = units;
    units += static_cast<uint32_t>(more);
  }
  // The tensor `unit` belongs to (the same in every lane).
  __device__ __forceinline__ uint32_t tensor_of(uint32_t unit) const {
    if constexpr (N == 1) return 0;
    uint32_t started = 0;
#pragma unroll
    for (uint32_t base = 0; base < static_cast<uint32_t>(N); base += kWave) {
      const uint32_t t = base + threadIdx.x % kWave;
      const bool starts = t < tensors && first[t < N ? t : 0] <= unit;
      started += static_cast<uint32_t>(__popcll(__ballot(starts)));
    }
    return started - 1;
  }
};

constexpr uint64_t kOwnLaunchBytes = uint64_t{64} << 20;

template <typename T>
struct AdamwEntry {
  T* parameter;
  const T* gradient;
  T* first;
  T* second;
  uint64_t count;
  double first_correction;
  double second_correction;
};

constexpr int kAdamwTensors = 64;

template <typename T, int N>
struct AdamwBatch {
  UnitMap<N> map;
  AdamwEntry<T> tensors[N];
};

// A single-wave workgroup updates a tile of 2 x 64 16-byte vectors of each of
// a tensor's arrays, issuing all eight loads of a lane (grouped by array)
// before its first store.  Measured on MI355X over 124M fp32 elements: two
// vectors per lane beat one (5.90 vs 5.76 TB/s) and four (5.47); a variant
// with the same traffic and no arithmetic runs no faster, so the double math
// is hidden.
constexpr int kAdamwUnroll = 2;
constexpr uint64_t kAdamwTile = static_cast<uint64_t>(kVectorThreads) * kAdamwUnroll;

template <typename T, int N, bool NT>
__global__ void __launch_bounds__(kVectorThreads)
    adamw_batch_kernel(AdamwBatch<T, N> batch, AdamwStep step) {
  using V = typename Vec16<T>::type;
  constexpr int W = Vec16<T>::width;
  constexpr int U = kAdamwUnroll;
  for (uint32_t unit = blockIdx.x; unit < batch.map.units; unit += gridDim.x) {
    const uint32_t t = batch.map.tensor_of(unit);
    const AdamwEntry<T> e = batch.tensors[t];
    step.first_correction = e.first_correction;
    step.second_correction = e.second_correction;
    const uint64_t vectors = e.count / W;
    V* p_v = reinterpret_cast<V*>(e.parameter);
    const V* g_v = reinterpret_cast<const V*>(e.gradient);
    V* m_v = reinterpret_cast<V*>(e.first);
    V* s_v = reinterpret_cast<V*>(e.second);
    const uint32_t tile = unit - batch.map.first[t];
    const uint64_t base = tile * kAdamwTile + threadIdx.x;
    V p[U], g[U], m[U], s[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const uint64_t i = base + static_cast<uint64_t>(u) * kVectorThreads;
      if (i < vectors) p[u] = stream_load(p_v + i);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const uint64_t i = base + static_cast<uint64_t>(u) * kVectorThreads;
      if (i < vectors) g[u] = stream_load(g_v + i);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const uint64_t i = base + static_cast<uint64_t>(u) * kVectorThreads;
      if (i < vectors) m[u] = stream_load(m_v + i);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const uint64_t i = base + static_cast<uint64_t>(u) * kVectorThreads;
      if (i < vectors) s[u] = stream_load(s_v + i);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const uint64_t i = base + static_cast<uint64_t>(u) * kVectorThreads;
      if (i >= vectors) continue;
#pragma unroll
      for (int k = 0; k < W; ++k) {
        T pk = vec_get<T>(p[u], k), mk = vec_get<T>(m[u], k), sk = vec_get<T>(s[u], k);
        adamw_element(pk, vec_get<T>(g[u], k), mk, sk, step);
        vec_set<T>(p[u], k, pk);
        vec_set<T>(m[u], k, mk);
        vec_set<T>(s[u], k, sk);
      }
      store_vector<NT>(m_v + i, m[u]);
      store_vector<NT>(s_v + i, s[u]);
      store_vector<NT>(p_v + i, p[u]);
    }
    if (tile == 0) {  // the count % W last elements
      const uint64_t i = vectors * W + threadIdx.x;
      if (i < e.count) {
        adamw_element(e.parameter[i], e.gradient[i], e.first[i], e.second[i], step);
      }
    }
  }
}

template <typename T>
__global__ void __launch_bounds__(kThreads)
    adamw_scalar_kernel(T* parameter, const T* gradient, T* first, T* second, uint64_t count,
                        AdamwStep step) {
  const uint64_t stride = static_cast<uint64_t>(gridDim.x) * kThreads;
  for (uint64_t i = static_cast<uint64_t>(blockIdx.x) * kThreads + threadIdx.x; i < count;
       i += stride) {
    adamw_element(parameter[i], gradient[i], first[i], second[i], step);
  }
}

uint64_t units_of(uint64_t vectors, uint64_t per_unit) {
  const uint64_t units = (vectors + per_unit - 1) / per_unit;
  return units == 0 ? 1 : units;
}

uint32_t unit_grid(uint32_t units) {
  return units > kMaxGrid ? static_cast<uint32_t>(kMaxGrid) : units;
}

// Collects tensors for launches of up to N: add() launches what is held when
// the next tensor does not fit, flush() what is left.  `Batch` holds `map`
// and arrays of N entries, `entry(batch, t)` fills slot t and
// `launch(batch, bytes)` enqueues, given the bytes the batch writes.
template <typename Batch, typename Launch>
class Collector {
 public:
  explicit Collector(Launch launch) : launch_(launch) {}
  template <typename Entry>
  void add(uint64_t units, uint64_t bytes, Entry entry) {
    if (!batch_.map.accepts(units)) flush();
    entry(batch_, batch_.map.tensors);
    batch_.map.append(units);
    bytes_ += bytes;
  }
  void flush() {
    if (batch_.map.tensors != 0) launch_(batch_, bytes_);
    batch_.map = {};
    bytes_ = 0;
  }

 private:
  Batch batch_;
  uint64_t bytes_ = 0;
  Launch launch_;
};

// Updates `tensor_count` tensors; one whose arrays are not all 16-byte
// aligned takes the scalar kernel.
template <typename T>
void launch_adamw(const SparHipAdamwTensor* tensors, uint64_t tensor_count, AdamwStep step,
                  const DeviceGuard& guard) {
  auto launch = [&]<int N>(const AdamwBatch<T, N>& batch, uint64_t bytes) {
    with_policy(stream_output(bytes), [&](auto nt) {
      adamw_batch_kernel<T, N, decltype(nt)::value>
          <<<unit_grid(batch.map.units), kVectorThreads, 0, guard.stream>>>(batch, step);
    });
  };
  Collector<AdamwBatch<T, kAdamwTensors>, decltype(launch)> shared(launch);
  Collector<AdamwBatch<T, 1>, decltype(launch)> own(launch);
  for (uint64_t k = 0; k < tensor_count; ++k) {
    const SparHipAdamwTensor& tensor = tensors[k];
    if (tensor.count == 0) continue;
    const AdamwEntry<T> entry{static_cast<T*>(tensor.parameter),
                              static_cast<const T*>(tensor.gradient),
                              static_cast<T*>(tensor.first_moment),
                              static_cast<T*>(tensor.second_moment),
                              tensor.count,
                              tensor.first_correction,
                              tensor.second_correction};
    const uint64_t units = units_of(tensor.count / Vec16<T>::width, kAdamwTile);
    if (!aligned16(entry.parameter) || !aligned16(entry.gradient) || !aligned16(entry.first) ||
        !aligned16(entry.second) || units > kIndex32Limit) {
      step.first_correction = entry.first_correction;
      step.second_correction = entry.second_correction;
      adamw_scalar_kernel<T><<<scalar_grid(entry.count, guard), kThreads, 0, guard.stream>>>(
          entry.parameter, entry.gradient, entry.first, entry.second, entry.count, step);
      continue;
    }
    const uint64_t bytes = tensor.count * sizeof(T);
    auto fill = [&](auto& batch, uint32_t t) { batch.tensors[t] = entry; };
    if (tensor_count == 1 || bytes >= kOwnLaunchBytes) {
      own.add(units, 3 * bytes, fill);
    } else {
      shared.add(units, 3 * bytes, fill);
    }
  }
  own.flush();
  shared.flush();
}

// ---------------------------------------------------------------- scaling

// training/gradients.cpp:107-111: v = (T)((double)v * factor).
template <typename T>
__device__ __forceinline__ T scaled(T value, double factor) {
  return static_cast<T>(static_cast<double>(value) * factor);
}

constexpr int kScaleTensors = 128;

template <typename T, int N>
struct ScaleBatch {
  UnitMap<N> map;
  T* values[N];
  uint64_t counts[N];
};

// A unit is one vector per lane of a single-wave workgroup.
template <typename T, int N, bool NT>
__global__ void __launch_bounds__(kVectorThreads)
    scale_batch_kernel(ScaleBatch<T, N> batch, double factor) {
  using V = typename Vec16<T>::type;
  constexpr int W = Vec16<T>::width;
  for (uint32_t unit = blockIdx.x; unit < batch.map.units; unit += gridDim.x) {
    const uint32_t t = batch.map.tensor_of(unit);
    T* values = batch.values[t];
    const uint64_t count = batch.counts[t];
    const uint64_t vectors = count / W;
    const uint32_t tile = unit - batch.map.first[t];
    V* v_v = reinterpret_cast<V*>(values);
    const uint64_t i = static_cast<uint64_t>(tile) * kVectorThreads + threadIdx.x;
    if (i < vectors) {
      V v = stream_load(v_v + i);
#pragma unroll
      for (int k = 0; k < W; ++k) vec_set<T>(v, k, scaled(vec_get<T>(v, k), factor));
      store_vector<NT>(v_v + i, v);
    }
    if (tile == 0) {  // the count % W last elements
      const uint64_t rest = vectors * W + threadIdx.x;
      if (rest < count) values[rest] = scaled(values[rest], factor);
    }
  }
}

template <typename T>
__global__ void __launch_bounds__(kThreads)
    scale_scalar_kernel(T* values, uint64_t count, double factor) {
  const uint64_t stride = static_cast<uint64_t>(gridDim.x) * kThreads;
  for (uint64_t i = static_cast<uint64_t>(blockIdx.x) * kThreads + threadIdx.x; i < count;
       i += stride) {
    values[i] = scaled(values[i], factor);
  }
}

template <typename T>
void launch_scale(void* const* values, const uint64_t* counts, uint64_t tensor_count,
                  double factor, const DeviceGuard& guard) {
  auto launch = [&]<int N>(const ScaleBatch<T, N>& batch, uint64_t bytes) {
    with_policy(stream_output(bytes), [&](auto nt) {
      scale_batch_kernel<T, N, decltype(nt)::value>
          <<<unit_grid(batch.map.units), kVectorThreads, 0, guard.stream>>>(batch, factor);
    });
  };
  Collector<ScaleBatch<T, kScaleTensors>, decltype(launch)> shared(launch);
  Collector<ScaleBatch<T, 1>, decltype(launch)> own(launch);
  for (uint64_t k = 0; k < tensor_count; ++k) {
    const uint64_t count = counts[k];
    if (count == 0) continue;
    T* data = static_cast<T*>(values[k]);
    const uint64_t units = units_of(count / Vec16<T>::width, kVectorThreads);
    if (!aligned16(data) || units > kIndex32Limit) {
      scale_scalar_kernel<T><<<scalar_grid(count, guard), kThreads, 0, guard.stream>>>(data, count,
                                                                                      factor);
      continue;
    }
    const uint64_t bytes = count * sizeof(T);
    auto fill = [&](auto& batch, uint32_t t) {
      batch.values[t] = data;
      batch.counts[t] = count;
    };
    if (tensor_count == 1 || bytes >= kOwnLaunchBytes) {
      own.add(units, bytes, fill);
    } else {
      shared.add(units, bytes, fill);
    }
  }
  own.flush();
  shared.flush();
}

// ----------------------------------------------------------- norm summary

// Exponent of a sum that holds no element yet: below every double's, so it
// never wins a max, and rescaling by it flushes only zeros.
constexpr int kNoExponent = -4096;

// Sum of squares of finite elements held as sum * 2^(2 * exponent), plus the
// largest finite magnitude and the infinity / NaN flags.
struct NormPartial {
  double sum;
  double maximum;
  int32_t exponent;
  int32_t flags;  // bit 0: an infinity was seen, bit 1: a NaN was seen
};

__device__ __forceinline__ NormPartial empty_partial() {
  return NormPartial{0.0, 0.0, kNoExponent, 0};
}

__device__ __forceinline__ NormPartial merge(NormPartial a, const NormPartial& b) {
  const int32_t e = a.exponent > b.exponent ? a.exponent : b.exponent;
  a.sum = ldexp(a.sum, 2 * (a.exponent - e)) + ldexp(b.sum, 2 * (b.exponent - e));
  a.exponent = e;
  a.maximum = fmax(a.maximum, b.maximum);
  a.flags |= b.flags;
  return a;
}

// One element into a lane's partial.  CAREFUL applies the reference's
// classification (gradients.cpp:30-40): infinities and NaNs set their flags
// and are left out of the sum and maximum.  The fast form omits it; a
// non-finite element then makes the lane's sum non-finite, which sends the
// lane to the careful form.
template <bool CAREFUL>
__device__ __forceinline__ void accumulate(NormPartial& p, float x) {
  // Squares of floats are exact in double and a sum of at most 2^64 of them
  // stays below 2^320: the exponent stays 0 and no rescaling is needed.
  float a = fabsf(x);
  if constexpr (CAREFUL) {
    if (x != x) p.flags |= 2;
    if (a == __builtin_huge_valf()) p.flags |= 1;
    if (!(a < __builtin_huge_valf())) a = 0.0f;
  }
  const double d = static_cast<double>(a);
  p.sum = fma(d, d, p.sum);
  p.maximum = fmax(p.maximum, d);
}

template <bool CAREFUL>
__device__ __forceinline__ void accumulate(NormPartial& p, double x) {
  double a = fabs(x);
  if constexpr (CAREFUL) {
    if (x != x) p.flags |= 2;
    if (a == __builtin_huge_val()) p.flags |= 1;
    if (!(a < __builtin_huge_val())) a = 0.0;
  }
  // v_frexp_exp: a = m * 2^e with m in [0.5, 1) for finite nonzero a.
  const int e = a == 0.0 ? kNoExponent : __builtin_amdgcn_frexp_exp(a);
  const int32_t top = p.exponent > e ? p.exponent : e;
  const double t = ldexp(a, -top);
  p.sum = fma(t, t, ldexp(p.sum, 2 * (p.exponent - top)));
  p.exponent = top;
  p.maximum = fmax(p.maximum, a);
}

// One lane's elements of [begin, end): 16-byte vectors strided by the block,
// two in flight (with the many short segments below, deeper unrolling
// measured no faster).
template <typename T, bool CAREFUL>
__device__ __forceinline__ NormPartial lane_summary(const T* gradient, uint64_t begin,
                                                    uint64_t end) {
  using V = typename Vec16<T>::type;
  constexpr int W = Vec16<T>::width;
  NormPartial p = empty_partial();
  if constexpr (sizeof(T) == 4) p.exponent = 0;
  const V* g_v = reinterpret_cast<const V*>(gradient);
  const uint64_t step = kThreads;
  uint64_t i = begin / W + threadIdx.x;
  const uint64_t stop = end / W;
  for (; i + step < stop; i += 2 * step) {
    const V v0 = stream_load(g_v + i);
    const V v1 = stream_load(g_v + i + step);
#pragma unroll
    for (int k = 0; k < W; ++k) accumulate<CAREFUL>(p, vec_get<T>(v0, k));
#pragma unroll
    for (int k = 0; k < W; ++k) accumulate<CAREFUL>(p, vec_get<T>(v1, k));
  }
  for (; i < stop; i += step) {
    const V v = stream_load(g_v + i);
#pragma unroll
    for (int k = 0; k < W; ++k) accumulate<CAREFUL>(p, vec_get<T>(v, k));
  }
  return p;
}

__device__ __forceinline__ NormPartial wave_merge(NormPartial p) {
#pragma unroll
  for (int lane_mask = kWave / 2; lane_mask > 0; lane_mask >>= 1) {
    NormPartial other;
    other.sum = __shfl_xor(p.sum, lane_mask, kWave);
    other.maximum = __shfl_xor(p.maximum, lane_mask, kWave);
    other.exponent = __shfl_xor(p.exponent, lane_mask, kWave);
    other.flags = __shfl_xor(p.flags, lane_mask, kWave);
    p = merge(p, other);
  }
  return p;
}

// Block partials as separate arrays, so that the combine reads them coalesced.
struct PartialArrays {
  double* sum;
  double* maximum;
  int32_t* exponent;
  int32_t* flags;
};

constexpr int kNormTensors = 128;

template <typename T, int N>
struct NormBatch {
  UnitMap<N> map;  // units: segments
  const T* gradients[N];
  uint64_t counts[N];
  uint64_t segments[N];  // elements of a segment
};

// Segment b of a gradient is its elements [b * segment, min((b + 1) * segment,
// count)) (segments are multiples of the vector width; the unaligned tail of
// the last vector goes to segment 0's first lanes); its partial is written at
// its unit.
template <typename T, int N>
__global__ void __launch_bounds__(kThreads)
    norm_partial_kernel(PartialArrays partials, NormBatch<T, N> batch) {
  constexpr int W = Vec16<T>::width;
  const uint32_t t = batch.map.tensor_of(blockIdx.x);
  const uint32_t b = blockIdx.x - batch.map.first[t];
  const T* gradient = batch.gradients[t];
  const uint64_t count = batch.counts[t];
  const uint64_t segment = batch.segments[t];
  const uint64_t body = count / W * W;
  const uint64_t begin = static_cast<uint64_t>(b) * segment;
  const uint64_t end = begin + segment < body ? begin + segment : body;
  NormPartial p = empty_partial();
  if (begin < end) {
    p = lane_summary<T, false>(gradient, begin, end);
    if (!(p.sum < __builtin_huge_val())) p = lane_summary<T, true>(gradient, begin, end);
  }
  if (b == 0 && body + threadIdx.x < count) {
    NormPartial q = empty_partial();
    if constexpr (sizeof(T) == 4) q.exponent = 0;
    accumulate<true>(q, gradient[body + threadIdx.x]);
    p = merge(p, q);
  }
  p = wave_merge(p);
  __shared__ NormPartial waves[kThreads / kWave];
  const int wave = threadIdx.x / kWave;
  if (threadIdx.x % kWave == 0) waves[wave] = p;
  __syncthreads();
  if (threadIdx.x == 0) {
    NormPartial total = waves[0];
#pragma unroll
    for (int w = 1; w < kThreads / kWave; ++w) total = merge(total, waves[w]);
    partials.sum[blockIdx.x] = total.sum;
    partials.maximum[blockIdx.x] = total.maximum;
    partials.exponent[blockIdx.x] = total.exponent;
    partials.flags[blockIdx.x] = total.flags;
  }
}

constexpr int kCombineThreads = 1024;
constexpr int kCombineWaves = kCombineThreads / kWave;
constexpr int kCombineBatch = 16;

// Which partials each workgroup of the combine takes, and where it writes.
struct NormOutputs {
  uint32_t first[kNormTensors];  // first partial of each gradient
  uint32_t parts[kNormTensors];
  uint32_t slots[kNormTensors];  // its summary
};

// Workgroup t combines gradient t's `parts` partials in a fixed order and
// writes its summary in the reference's form (SparCudaNormSummary): scale = the largest finite
// magnitude, scaled_sum_squares = sum of (x / scale)^2; {0, 1} when no finite
// nonzero element was seen, as the reference's initial state.  RESCALE (fp64
// partials): two passes, the common exponent, maximum and flags first, then
// every partial's sum rescaled to that exponent, so neither pass is a chain
// of dependent merges.  fp32 partials all have exponent 0 (or hold nothing),
// so the rescale is the identity and one pass adds the same values in the
// same order: the same bits, one round trip to the partials instead of two.
template <bool RESCALE>
__global__ void __launch_bounds__(kCombineThreads)
    norm_combine_kernel(SparHipNormSummary* summaries, PartialArrays partials,
                        NormOutputs outputs) {
  const uint64_t parts = outputs.parts[blockIdx.x];
  const uint32_t offset = outputs.first[blockIdx.x];
  partials.sum += offset;
  partials.maximum += offset;
  partials.exponent += offset;
  partials.flags += offset;
  __shared__ int32_t wave_top[kCombineWaves];
  __shared__ int32_t wave_flags[kCombineWaves];
  __shared__ double wave_maximum[kCombineWaves];
  __shared__ double wave_total[kCombineWaves];
  const int lane = threadIdx.x % kWave;
  const int wave = threadIdx.x / kWave;
  // fp32 partials that hold elements all have exponent 0, so theirs is 0
  int32_t top = RESCALE ? kNoExponent : 0;
  int32_t flags = 0;
  double maximum = 0.0;
  double sum = 0.0;
  // The partials come from every XCD: each batch issues all of a thread's
  // loads before using any, so a pass costs about one round trip.
  for (uint64_t base = threadIdx.x; base < parts; base += kCombineThreads * kCombineBatch) {
    int32_t e[kCombineBatch], f[kCombineBatch];
    double m[kCombineBatch];
    double v[RESCALE ? 1 : kCombineBatch];
#pragma unroll
    for (int k = 0; k < kCombineBatch; ++k) {
      const uint64_t i = base + static_cast<uint64_t>(k) * kCombineThreads;
      const bool in = i < parts;
      if constexpr (RESCALE) e[k] = in ? partials.exponent[i] : kNoExponent;
      m[k] = in ? partials.maximum[i] : 0.0;
      f[k] = in ? partials.flags[i] : 0;
      if constexpr (!RESCALE) v[k] = in ? partials.sum[i] : 0.0;
    }
#pragma unroll
    for (int k = 0; k < kCombineBatch; ++k) {
      if constexpr (RESCALE) top = max(top, e[k]);
      maximum = fmax(maximum, m[k]);
      flags |= f[k];
      if constexpr (!RESCALE) sum += v[k];
    }
  }
#pragma unroll
  for (int lane_mask = kWave / 2; lane_mask > 0; lane_mask >>= 1) {
    top = max(top, __shfl_xor(top, lane_mask, kWave));
    maximum = fmax(maximum, __shfl_xor(maximum, lane_mask, kWave));
    flags |= __shfl_xor(flags, lane_mask, kWave);
  }
  if (lane == 0) {
    wave_top[wave] = top;
    wave_maximum[wave] = maximum;
    wave_flags[wave] = flags;
  }
  __syncthreads();
  top = wave_top[0];
  maximum = wave_maximum[0];
  flags = wave_flags[0];
#pragma unroll
  for (int w = 1; w < kCombineWaves; ++w) {
    top = max(top, wave_top[w]);
    maximum = fmax(maximum, wave_maximum[w]);
    flags |= wave_flags[w];
  }
  if constexpr (RESCALE) {
    for (uint64_t base = threadIdx.x; base < parts; base += kCombineThreads * kCombineBatch) {
      int32_t e[kCombineBatch];
      double v[kCombineBatch];
#pragma unroll
      for (int k = 0; k < kCombineBatch; ++k) {
        const uint64_t i = base + static_cast<uint64_t>(k) * kCombineThreads;
        const bool in = i < parts;
        e[k] = in ? partials.exponent[i] : top;
        v[k] = in ? partials.sum[i] : 0.0;
      }
#pragma unroll
      for (int k = 0; k < kCombineBatch; ++k) sum += ldexp(v[k], 2 * (e[k] - top));
    }
  }
  sum = wave_sum(sum);
  if (lane == 0) wave_total[wave] = sum;
  __syncthreads();
  if (threadIdx.x == 0) {
    double total = wave_total[0];
#pragma unroll
    for (int w = 1; w < kCombineWaves; ++w) total += wave_total[w];
    SparHipNormSummary out;
    if (maximum == 0.0) {
      out.scale = 0.0;
      out.scaled_sum_squares = 1.0;
    } else {
      // maximum = r * 2^top with r in [0.5, 1) for fp64 input (top = 0 for
      // fp32); sum * 2^(2 top) / maximum^2 = sum / r^2.
      const double r = ldexp(maximum, -top);
      out.scale = maximum;
      out.scaled_sum_squares = total / r / r;
    }
    out.has_infinity = flags & 1;
    out.has_nan = (flags >> 1) & 1;
    summaries[outputs.slots[blockIdx.x]] = out;
  }
}

// The summaries of `tensor_count` gradients (an empty one's is the combine of
// no partials) into device_summaries[0 ...].
template <typename T, int N>
hipError_t launch_norm_summaries(SparHipNormSummary* device_summaries,
                                 const void* const* gradients, const uint64_t* counts,
                                 uint64_t tensor_count, int device, const DeviceGuard& guard) {
  constexpr int W = Vec16<T>::width;
  // Segments of at least four vectors per lane and up to 64 blocks per CU:
  // over 124M fp32 elements 16384 short segments read at 6.7 TB/s where
  // 2048 long ones reach 6.1 TB/s.
  const uint64_t min_segment = static_cast<uint64_t>(kThreads) * W * 4;
  const uint64_t max_blocks = static_cast<uint64_t>(guard.multiprocessors) * 64;
  NormBatch<T, N> batch;
  NormOutputs outputs{};
  uint32_t summaries = 0;
  auto flush = [&]() -> hipError_t {
    if (summaries == 0) return hipSuccess;
    const uint64_t blocks = batch.map.units;
    void* scratch = nullptr;
    if (blocks != 0) {
      const hipError_t error = scratch_allocate(&scratch, blocks * 24, device);
      if (error != hipSuccess) return error;
    }
    char* bytes = static_cast<char*>(scratch);
    const PartialArrays partials{reinterpret_cast<double*>(bytes),
                                 reinterpret_cast<double*>(bytes + 8 * blocks),
                                 reinterpret_cast<int32_t*>(bytes + 16 * blocks),
                                 reinterpret_cast<int32_t*>(bytes + 20 * blocks)};
    if (blocks != 0) {
      norm_partial_kernel<T, N>
          <<<batch.map.units, kThreads, 0, guard.stream>>>(partials, batch);
    }
    norm_combine_kernel<(sizeof(T) > 4)>
        <<<summaries, kCombineThreads, 0, guard.stream>>>(device_summaries, partials, outputs);
    scratch_release(scratch, device);  // stream-ordered reuse
    batch.map = {};
    summaries = 0;
    return hipGetLastError();
  };
  for (uint64_t k = 0; k < tensor_count; ++k) {
    const uint64_t count = counts[k];
    const uint64_t body = count / W * W;
    uint64_t blocks = (body + min_segment - 1) / min_segment;
    if (blocks > max_blocks) blocks = max_blocks;
    if (blocks == 0) blocks = 1;
    uint64_t segment = (body + blocks - 1) / blocks;
    segment = (segment + W - 1) / W * W;
    if (segment == 0) segment = W;
    blocks = count == 0 ? 0 : body == 0 ? 1 : (body + segment - 1) / segment;
    if (summaries == static_cast<uint32_t>(N)) {
      if (const hipError_t error = flush(); error != hipSuccess) return error;
    }
    outputs.first[summaries] = batch.map.units;
    outputs.parts[summaries] = static_cast<uint32_t>(blocks);
    outputs.slots[summaries] = static_cast<uint32_t>(k);
    ++summaries;
    if (blocks != 0) {
      const uint32_t t = batch.map.tensors;
      batch.gradients[t] = static_cast<const T*>(gradients[k]);
      batch.counts[t] = count;
      batch.segments[t] = segment;
      batch.map.append(blocks);
    }
  }
  return flush();
}

hipError_t launch_norm_summaries(SparHipNormSummary* device_summaries,
                                 const void* const* gradients, const uint64_t* counts,
                                 uint64_t tensor_count, int dtype, int device,
                                 const DeviceGuard& guard) {
  auto run = [&]<typename T>(T) {
    return tensor_count == 1
               ? launch_norm_summaries<T, 1>(device_summaries, gradients, counts, 1, device, guard)
               : launch_norm_summaries<T, kNormTensors>(device_summaries, gradients, counts,
                                                        tensor_count, device, guard);
  };
  return dtype == SPAR_HIP_FLOAT32 ? run(float{}) : run(double{});
}

}  // namespace
}  // namespace spar_hip

using namespace spar_hip;

extern "C" SparHipStatus spar_hip_launch_adamw_batch(const SparHipAdamwTensor* tensors,
                                                     uint64_t tensor_count, int dtype,
                                                     double learning_rate, double beta1,
                                                     double beta2, double epsilon,
                                                     double weight_decay, int device) {
  if (!valid_float_dtype(dtype) || (tensor_count != 0 && tensors == nullptr)) return invalid();
  bool empty = true;
  for (uint64_t k = 0; k < tensor_count; ++k) {
    const SparHipAdamwTensor& t = tensors[k];
    if (t.count == 0) continue;
    empty = false;
    if (t.parameter == nullptr || t.gradient == nullptr || t.first_moment == nullptr ||
        t.second_moment == nullptr) {
      return invalid();
    }
  }
  if (empty) return ok();
  DeviceGuard guard;
  if (enter(device, guard) != hipSuccess) return runtime(guard.error);
  AdamwStep step;
  step.learning_rate = learning_rate;
  step.beta1 = beta1;
  step.beta2 = beta2;
  step.epsilon = epsilon;
  step.first_correction = 1.0;  // each tensor's own
  step.second_correction = 1.0;
  step.one_minus_beta1 = 1.0 - beta1;
  step.one_minus_beta2 = 1.0 - beta2;
  step.decay_factor = 1.0 - learning_rate * weight_decay;
  if (dtype == SPAR_HIP_FLOAT32) {
    launch_adamw<float>(tensors, tensor_count, step, guard);
  } else {
    launch_adamw<double>(tensors, tensor_count, step, guard);
  }
  return finish(guard);
}

extern "C" SparHipStatus spar_hip_launch_adamw(void* parameter, const void* gradient,
                                               void* first_moment, void* second_moment,
                                               uint64_t count, int dtype, double learning_rate,
                                               double beta1, double beta2, double epsilon,
                                               double weight_decay, double first_correction,
                                               double second_correction, int device) {
  const SparHipAdamwTensor tensor{parameter,     gradient, first_moment,
                                  second_moment, count,    first_correction,
                                  second_correction};
  return spar_hip_launch_adamw_batch(&tensor, 1, dtype, learning_rate, beta1, beta2, epsilon,
                                     weight_decay, device);
}

extern "C" SparHipStatus spar_hip_launch_scale_in_place_batch(void* const* values,
                                                              const uint64_t* counts,
                                                              uint64_t tensor_count, int dtype,
                                                              double factor, int device) {
  if (!valid_float_dtype(dtype) || !isfinite(factor) ||
      (tensor_count != 0 && (values == nullptr || counts == nullptr))) {
    return invalid();
  }
  bool empty = true;
  for (uint64_t k = 0; k < tensor_count; ++k) {
    if (counts[k] == 0) continue;
    empty = false;
    if (values[k] == nullptr) return invalid();
  }
  if (empty) return ok();
  DeviceGuard guard;
  if (enter(device, guard) != hipSuccess) return runtime(guard.error);
  if (dtype == SPAR_HIP_FLOAT32) {
    launch_scale<float>(values, counts, tensor_count, factor, guard);
  } else {
    launch_scale<double>(values, counts, tensor_count, factor, guard);
  }
  return finish(guard);
}

extern "C" SparHipStatus spar_hip_launch_scale_in_place(void* values, uint64_t count, int dtype,
                                                        double factor, int device) {
  return spar_hip_launch_scale_in_place_batch(&values, &count, 1, dtype, factor, device);
}

extern "C" SparHipStatus spar_hip_launch_gradient_norm_summaries(SparHipNormSummary* summaries,
                                                                 const void* const* gradients,
                                                                 const uint64_t* counts,
                                                                 uint64_t tensor_count, int dtype,
                                                                 int device) {
  if (!valid_float_dtype(dtype) ||
      (tensor_count != 0 &&
       (summaries == nullptr || gradients == nullptr || counts == nullptr))) {
    return invalid();
  }
  for (uint64_t k = 0; k < tensor_count; ++k) {
    if (counts[k] != 0 && gradients[k] == nullptr) return invalid();
  }
  if (tensor_count == 0) return ok();
  DeviceGuard guard;
  if (enter(device, guard) != hipSuccess) return runtime(guard.error);
  const hipError_t error = launch_norm_summaries(summaries, gradients, counts, tensor_count, dtype,
                                                 device, guard);
  return error == hipSuccess ? ok() : runtime(error);
}

extern "C" SparHipStatus spar_hip_launch_gradient_norm_summary(SparHipNormSummary* summary,
                                                               const void* gradient,
                                                               uint64_t count, int dtype,
                                                               int device) {
  return spar_hip_launch_gradient_norm_summaries(summary, &gradient, &count, 1, dtype, device);
}

extern "C" SparHipStatus spar_hip_gradient_norm_summary(SparHipNormSummary* host_summary,
                                                        const void* gradient, uint64_t count,
                                                        int dtype, int device) {
  if (host_summary == nullptr || !valid_float_dtype(dtype) ||
      (count != 0 && gradient == nullptr)) {
    return invalid();
  }
  *host_summary = SparHipNormSummary{0.0, 1.0, 0, 0};
  if (count == 0) return ok();
  DeviceGuard guard;
  if (enter(device, guard) != hipSuccess) return runtime(guard.error);
  void* scratch = nullptr;
  hipError_t error = scratch_allocate(&scratch, sizeof(SparHipNormSummary), device);
  if (error != hipSuccess) return runtime(error);
  SparHipNormSummary* device_summary = static_cast<SparHipNormSummary*>(scratch);
  error = launch_norm_summaries(device_summary, &gradient, &count, 1, dtype, device, guard);
  SparHipStatus status = error == hipSuccess ? ok() : runtime(error);
  if (status.code == 0) {
    status = spar_hip_copy_device_to_host(host_summary, device_summary,
                                          sizeof(SparHipNormSummary), device);
  }
  scratch_release(scratch, device);
  return status;
}
