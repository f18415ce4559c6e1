// Cross-entropy statistics of full logits rows (gfx950): the fallback used when the logits
// exist anyway. Reproduces solution/lm_head_loss.py:54-96 (lm_head_xent_rows_kernel):
//   per row: M = max z, S = sum e^{z-M}, D = sum e^{z-M} z, lse = M + ln S,
//   loss = label ? lse - z[t] : 0, entropy = lse - D/S, correct = label && argmax == t
//   (first index of the maximum), and optionally the row overwritten by
//   round((softmax - onehot) * grad_scale), zero for unlabelled rows.
//
// One workgroup per row; each lane keeps an online (max, sum, dot, argmax) state over its columns,
// eight at a time: the eight's maximum first, so that a value costs one exponential and the state
// is rescaled only when its maximum moves. At the end the row's maximum is found, every lane
// rescales to it once and the sums are added. Chunks start at 16-byte boundaries of memory, whatever
// the row's own alignment (16-byte loads); only a row's first and last chunk may be partial and go
// element by element, their missing columns as -inf. e^x is computed as 2^(x log2 e) on v_exp_f32,
// ln as log2 * ln 2 on v_log_f32.
//
// A -inf logit adds nothing, a NaN or +inf makes the row's loss NaN. A state whose scale is 0
// against a larger maximum drops its dot: values near the type's lowest may have taken it to -inf.
//
// What bounds it: memory, a read of the row, and with the gradient another and a write. 151936 bf16
// logits, us with / without the gradient: 1000 rows 141 / 55 (6.5 / 5.6 TB/s; one value a step and
// two exponentials a value: 638 / 302), 300 rows 63 / 29 (420 / 209), 4096 rows of 5000 25 / 14
// (42 / 25); 300 rows of 151935 64 / 29 (417 / 208).
#include "common.h"

#include "softmax_state.h"
#include "vec.h"

namespace {

// Long rows take 1024 lanes: a row is a serial chain of loads, and a row's second reading finds more
// of it in the L2 the fewer rows are under way (151936 bf16 columns, us with gradient, 1024 / 256
// lanes: 511 rows 69 / 97, 1000 rows 141 / 159, 4000 rows 562 / 715). Shorter ones take them only
// while too few rows are there to fill the CUs (256 rows of 32768 14.6 / 17.2, 2000 rows 68 / 64, 4096
// rows of 24576 107 / 88: the lanes' start and merge count).
constexpr int64_t kWideCols = 65536;
constexpr int64_t kFewRowsWideCols = 32768;
constexpr int64_t kFewRows = 512;

constexpr float kLowest = -3.402823466e38f;

// A lane's walk over its chunks of a row of n_cols values at z: full(c) and full2(c) for one and two
// whole chunks (columns c .. c + 7, and kStep further), part(c) for one that reaches past an end.
template <typename T, int THREADS, typename Full2, typename Full, typename Part>
__device__ __forceinline__ void walk_row(const T* z, int64_t n_cols, Full2 full2, Full full,
                                         Part part) {
  constexpr int64_t kStep = THREADS * 8;
  const int lead = static_cast<int>(reinterpret_cast<uintptr_t>(z) % 16 / sizeof(T));
  int64_t c = static_cast<int64_t>(threadIdx.x) * 8 - lead;
  if (c < 0) {
    part(c);
    c += kStep;
  }
  for (; c + kStep + 8 <= n_cols; c += 2 * kStep) full2(c);
  for (; c + 8 <= n_cols; c += kStep) full(c);
  if (c < n_cols) part(c);
}

template <typename T, int THREADS>
__global__ __launch_bounds__(THREADS) void xent_rows_kernel(T* __restrict__ logits,
                                                            int64_t row_stride,
                                                            const int64_t* __restrict__ target,
                                                            float* __restrict__ loss,
                                                            float* __restrict__ entropy,
                                                            int32_t* __restrict__ correct,
                                                            int64_t n_cols, int write_grad,
                                                            float grad_scale) {
  using V = cm::Vec8<T, true>;
  constexpr int kStep = THREADS * 8;
  constexpr int kWaves = THREADS / cm::kWave;
  const int64_t row = blockIdx.x;
  T* z = logits + row * row_stride;
  cm::SoftmaxState st = cm::SoftmaxState::empty();
  auto push8 = [&](const float (&v)[8], int64_t c) {
    float m = v[0];
#pragma unroll
    for (int i = 1; i < 8; ++i) m = fmaxf(m, v[i]);
    if (m > st.max) {
      const float r = cm::exp_f(st.max - m);  // 0 while the state is empty
      st.sum *= r;
      st.dot = r == 0.0f ? 0.0f : st.dot * r;
      st.max = m;
      int first = 0;
#pragma unroll
      for (int i = 7; i >= 0; --i) first = v[i] == m ? i : first;
      st.best = c + first;
    }
    const float ref = fmaxf(st.max, kLowest);  // finite while only -inf has been seen
    float e[8], d[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      e[i] = cm::exp_f(v[i] - ref);
      d[i] = e[i] * fmaxf(v[i], kLowest);  // 0 for -inf
    }
#pragma unroll
    for (int n = 4; n > 0; n /= 2) {
#pragma unroll
      for (int i = 0; i < n; ++i) {
        e[i] += e[i + n];
        d[i] += d[i + n];
      }
    }
    st.sum += e[0];
    st.dot += d[0];
  };
  walk_row<T, THREADS>(
      z, n_cols,
      [&](int64_t c) {
        float a[8], b[8];
        V::load(z + c, a);
        V::load(z + c + kStep, b);
        push8(a, c);
        push8(b, c + kStep);
      },
      [&](int64_t c) {
        float a[8];
        V::load(z + c, a);
        push8(a, c);
      },
      [&](int64_t c) {
        float a[8];
#pragma unroll
        for (int i = 0; i < 8; ++i)
          a[i] = c + i >= 0 && c + i < n_cols ? cm::to_f32(z[c + i]) : -__builtin_huge_valf();
        push8(a, c);
      });

  // the row's maximum and its first index, then the sums at that maximum
  __shared__ float s_max[kWaves], s_sum[kWaves], s_dot[kWaves];
  __shared__ int64_t s_best[kWaves];
  const int wave = threadIdx.x / cm::kWave;
  const bool first_lane = threadIdx.x % cm::kWave == 0;
  float row_max = st.max;
  int64_t best = st.best;
  auto take = [&](float m, int64_t i) {
    if (m > row_max || (m == row_max && i < best)) {
      row_max = m;
      best = i;
    }
  };
#pragma unroll
  for (int off = 32; off > 0; off >>= 1)
    take(__shfl_xor(row_max, off, cm::kWave), __shfl_xor(best, off, cm::kWave));
  if (first_lane) {
    s_max[wave] = row_max;
    s_best[wave] = best;
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kWaves; ++i) take(s_max[i], s_best[i]);
  const float r = cm::exp_f(st.max - row_max);  // NaN where a row holds +inf or only -inf and NaN
  float sum = st.sum * r;
  float dot = r == 0.0f ? 0.0f : st.dot * r;
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    sum += __shfl_xor(sum, off, cm::kWave);
    dot += __shfl_xor(dot, off, cm::kWave);
  }
  if (first_lane) {
    s_sum[wave] = sum;
    s_dot[wave] = dot;
  }
  __syncthreads();
  const int w = threadIdx.x % kWaves;
  sum = s_sum[w];
  dot = s_dot[w];
#pragma unroll
  for (int off = kWaves / 2; off > 0; off >>= 1) {
    sum += __shfl_xor(sum, off, cm::kWave);
    dot += __shfl_xor(dot, off, cm::kWave);
  }

  const int64_t t = target[row];
  const bool labelled = t != -100;
  // A label outside [0, n_cols) is not read: its loss is NaN.
  const bool in_range = t >= 0 && t < n_cols;
  const float lse = row_max + cm::log_f(sum);
  if (threadIdx.x == 0) {
    const float zt = in_range ? cm::to_f32(z[t]) : __builtin_nanf("");
    loss[row] = labelled ? lse - zt : 0.0f;
    entropy[row] = lse - dot / sum;
    correct[row] = labelled && best == t ? 1 : 0;
  }
  if (write_grad) {
    __syncthreads();  // every lane has read its logits (and z[t]) before any is overwritten
    auto grad8 = [&](float (&v)[8], int64_t c) {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float p = cm::exp_f(v[i] - lse);
        v[i] = labelled ? (c + i == t ? p - 1.0f : p) * grad_scale : 0.0f;
      }
    };
    walk_row<T, THREADS>(
        z, n_cols,
        [&](int64_t c) {
          float a[8] = {}, b[8] = {};
          if (labelled) {
            V::load(z + c, a);
            V::load(z + c + kStep, b);
          }
          grad8(a, c);
          grad8(b, c + kStep);
          V::store(z + c, a);
          V::store(z + c + kStep, b);
        },
        [&](int64_t c) {
          float a[8];
          V::load(z + c, a);
          grad8(a, c);
          V::store(z + c, a);
        },
        [&](int64_t c) {
          float a[8];
#pragma unroll
          for (int i = 0; i < 8; ++i) a[i] = c + i >= 0 && c + i < n_cols ? cm::to_f32(z[c + i]) : 0.0f;
          grad8(a, c);
#pragma unroll
          for (int i = 0; i < 8; ++i)
            if (c + i >= 0 && c + i < n_cols) z[c + i] = cm::from_f32<T>(a[i]);
        });
  }
}

}  // namespace

extern "C" int cm_xent_rows(void* logits, int logits_dtype, int64_t row_stride,
                            const int64_t* target, float* loss, float* entropy, int32_t* correct,
                            int64_t n_rows, int64_t n_cols, int write_grad, float grad_scale,
                            void* stream) {
  CM_CHECK_ARG(n_rows >= 0 && n_cols > 0 && row_stride >= n_cols);
  if (n_rows == 0) return 0;
  CM_CHECK_ARG(logits && target && loss && entropy && correct);
  CM_CHECK_ARG(n_rows <= 0x7fffffff);
  hipStream_t s = static_cast<hipStream_t>(stream);
  const bool wide = n_cols >= (n_rows < kFewRows ? kFewRowsWideCols : kWideCols);
  CM_FLOAT_SWITCH(logits_dtype, T, {
    const auto kernel = wide ? xent_rows_kernel<T, 1024> : xent_rows_kernel<T, 256>;
    hipLaunchKernelGGL(kernel, dim3(static_cast<uint32_t>(n_rows)), dim3(wide ? 1024 : 256), 0, s,
                       static_cast<T*>(logits), row_stride, target, loss, entropy, correct, n_cols,
                       write_grad, grad_scale);
  });
  return cm::launch_status();
}
