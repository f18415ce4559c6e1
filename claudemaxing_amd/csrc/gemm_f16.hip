// fp16 linear layers that share an input, on expanded weights (gfx950): the q, k and v projections of
// an attention block after their NF4 weights were expanded into one [N, K] array, N = N_0 + N_1 + ..
//   forward   Y_i[m][n] = fp16(sum_k X[m][k] W_i[n][k] (+ b_i[n]))      (cm_linear_f16_fwd)
//   backward  dX[m][k] = fp16(sum_i sum_n G_i[m][n] W_i[n][k])          (cm_linear_f16_bwd)
// with fp32 sums, rounded once. The forward reads the weight by rows, the backward as stored, k-major
// (its contraction runs over the weight rows), through transposing LDS reads (gemm_lds.h).
//
// What bounds it: at a training step's 1276 tokens the outputs are 160 tiles of 128 x 128 (forward,
// contractions of 24 stages of 64 columns) or 240 of 128 x 64 (backward, 32 stages) on 256 CUs, one
// workgroup each (the rings take 128 and 96 KiB of a CU's LDS), each a serial chain of stages that take
// ~0.25 us of matrix-core time: latency, so the loads run two stages ahead and the fragments most of a
// stage (gemm_lds_small). Measured against the weights expanded inside the GEMM (nf4_gemm.hip), q/k/v
// of 1536 -> 1536 + 256 + 256, us forward / backward, the expansion of the three weights (~5 us alone,
// less among a layer's others) not counted: 65 tokens 8.8 / 14.0 against 28 / 21; 1276 15.1 / 16.4
// against 30 / 35; 8192 (256 x 256 tiles) 52 / 56 against 90 / 115.
#include "gemm_lds.h"
#include "nf4_tiles.h"

namespace {

using cm::gemm::floatx16;
using cm::gemm::KMajor;
using cm::gemm::RowMajor;
using cm::gemm::SegRows;

constexpr int kMaxOut = 3;

// The outputs, side by side along n: output s holds columns first[s] .. first[s + 1] - 1 (multiples
// of 64), rounded to fp16 after the bias (null: none).
struct Outputs {
  _Float16* p[kMaxOut];
  int64_t ld[kMaxOut];
  const _Float16* bias[kMaxOut];
  int first[kMaxOut];  // an unused output's is past N
  // the pick of column n's output, by selects (an index into the arrays would put them in memory)
  template <class T>
  __device__ __forceinline__ T of(int n, const T (&v)[kMaxOut]) const {
    const T v0 = v[0], v1 = v[1], v2 = v[2];
    const T a = n >= first[1] ? v1 : v0;
    return n >= first[2] ? v2 : a;
  }
};

// fp16(acc + bias) through the LDS: the accumulators lie 32 columns of 2 bytes at a time, the stores
// are 16 bytes per lane.
template <int BM, int BN, int WM, int WN>
struct EpiHalf {
  Outputs out;
  int M, N, m0, n0;
  template <int TM, int TN>
  __device__ __forceinline__ void prepare(int, int, int) {}
  template <int TM, int TN>
  __device__ __forceinline__ void start(floatx16 (&acc)[TM][TN], int mb, int nb, int lane) {
    cm::gemm::ZeroStart::start<TM, TN>(acc, mb, nb, lane);
  }
  template <int TM, int TN>
  __device__ __forceinline__ void started(floatx16 (&)[TM][TN]) {}
  template <int TM, int TN>
  __device__ __forceinline__ void apply(floatx16 (&acc)[TM][TN], int mb, int nb, int lane,
                                        uint4* lds) const {
    constexpr int kPitch = BN + 8;  // fp16 per staged row: 16-byte rows that start 4 banks apart
    constexpr int kThreads = WM * WN * cm::kWave;
    _Float16* tile = reinterpret_cast<_Float16*>(lds);
    // biases of the lane's columns, one 32-column accumulator tile at a time (inside one output)
    float bv[TN];
#pragma unroll
    for (int nt = 0; nt < TN; ++nt) {
      const int n = nb + nt * 32;
      const _Float16* b = out.of(n, out.bias);
      const int at = n - out.of(n, out.first) + lane % 32;
      bv[nt] = b != nullptr && n < N ? static_cast<float>(b[at]) : 0.0f;
    }
    cm::gemm::lds_barrier();  // every wavefront is done with the operand tiles
#pragma unroll
    for (int mt = 0; mt < TM; ++mt)
#pragma unroll
      for (int nt = 0; nt < TN; ++nt)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int row = mb - m0 + mt * 32 + (r / 4) * 8 + (lane / 32) * 4 + r % 4;
          tile[row * kPitch + nb - n0 + nt * 32 + lane % 32] =
              static_cast<_Float16>(acc[mt][nt][r] + bv[nt]);
        }
    cm::gemm::lds_barrier();
    constexpr int kChunks = BN / 8;
#pragma unroll 4
    for (int c = threadIdx.x; c < BM * kChunks; c += kThreads) {
      const int row = c / kChunks, n = n0 + c % kChunks * 8;
      if (m0 + row >= M || n >= N) continue;
      _Float16* const p = out.of(n, out.p) + (m0 + row) * out.of(n, out.ld);
      *reinterpret_cast<uint4*>(p + (n - out.of(n, out.first))) =
          *reinterpret_cast<const uint4*>(tile + row * kPitch + (n - n0));
    }
  }
};

// SMALL: gemm_lds_small on SA ring stages; SLICED: with its sums in slices
template <int BM_, int BN_, int WM_, int WN_, int SA_, int SB_, int OCC_, bool SMALL_,
          bool SLICED_ = false>
struct Cfg {
  static constexpr int BM = BM_, BN = BN_, WM = WM_, WN = WN_, SA = SA_, SB = SB_, kOcc = OCC_;
  static constexpr bool kSmall = SMALL_, kSliced = SLICED_;
  static constexpr int kThreads = WM * WN * cm::kWave;
  static constexpr int kLds = (SA * BM + SB * BN) * 8;
  static_assert(kLds * 16 >= BM * (BN + 8) * 2, "the epilogue's tile fits the operands' rings");
};
template <bool SLICED>
using Narrow = Cfg<128, 64, 2, 2, 4, 4, 1, true, SLICED>;
template <bool SLICED>
using Small = Cfg<128, 128, 2, 2, 4, 4, 1, true, SLICED>;
using Large = Cfg<256, 256, 2, 4, 3, 2, 2, false>;

template <class C, class SrcA, class SrcB>
__global__ __launch_bounds__(C::kThreads, C::kOcc) void linear_f16_kernel(SrcA a, SrcB b, Outputs out,
                                                                          int M, int N, int K,
                                                                          int remap, int slices) {
  __shared__ uint4 lds[C::kLds];
  int tm, tn;
  cm::gemm::tile_of(static_cast<int>(blockIdx.x), static_cast<int>(gridDim.x),
                    (N + C::BN - 1) / C::BN, remap, tm, tn);
  using Epi = EpiHalf<C::BM, C::BN, C::WM, C::WN>;
  Epi epi{out, M, N, tm * C::BM, tn * C::BN};
  if constexpr (C::kSmall) {
    cm::gemm::gemm_lds_small<C::BM, C::BN, C::WM, C::WN, C::SA, C::kSliced>(
        a, b, 0, K, tm, tn, epi, lds, slices);
  } else {
    cm::gemm::gemm_lds<C::BM, C::BN, C::WM, C::WN, C::SA, C::SB, SrcA, SrcB, Epi, cm::gemm::PlainA,
                       cm::gemm::kEdgeNever>(a, b, 0, K, tm, tn, epi, lds);
  }
}

template <class C, class SrcA, class SrcB>
int launch(const SrcA& a, const SrcB& b, const Outputs& out, int M, int N, int K, int slices,
           hipStream_t s) {
  const int64_t tiles = static_cast<int64_t>((M + C::BM - 1) / C::BM) * ((N + C::BN - 1) / C::BN);
  CM_CHECK_ARG(tiles <= 0x7fffffff);
  hipLaunchKernelGGL((linear_f16_kernel<C, SrcA, SrcB>), dim3(static_cast<unsigned>(tiles)),
                     dim3(C::kThreads), 0, s, a, b, out, M, N, K, tiles % 8 == 0 ? 1 : 0, slices);
  return cm::launch_status();
}

// The tile by the rounds of 256 workgroups (one per CU) an M x N output takes: 128 x 64 while one round
// of it holds the output (q/k/v forward at 640 tokens 11.6 us against 14.0 on 128 x 128; at 1276, two
// rounds, 20.4 against 15.1); 256 x 256 where its rounds, three and a bit times as long, are at most a
// third of 128 x 128's (8192 tokens: one round, 52 us, against four, 62; 4096: one against two, 41
// against 31); else 128 x 128.
int64_t rounds(int64_t M, int64_t N, int64_t bm, int64_t bn) {
  return ((M + bm - 1) / bm * ((N + bn - 1) / bn) + 255) / 256;
}

template <bool SLICED, class SrcA, class SrcB>
int launch_best(const SrcA& a, const SrcB& b, const Outputs& out, int M, int N, int K, int slices,
                hipStream_t s) {
  if (rounds(M, N, 128, 64) <= 1) return launch<Narrow<SLICED>>(a, b, out, M, N, K, slices, s);
  // 256 x 256 tiles sum in one slice (their accumulators leave no registers for a second set); more
  // than 512 tiles of 128 x 128, which they need, are never split
  if constexpr (!SLICED) {
    if (rounds(M, N, 256, 256) * 3 <= rounds(M, N, 128, 128))
      return launch<Large>(a, b, out, M, N, K, slices, s);
  }
  return launch<Small<SLICED>>(a, b, out, M, N, K, slices, s);
}

// Slices in which the input gradient of M rows is summed over its contraction of `stages` 64-column
// stages: those the NF4-fused GEMM splits it into (nf4_tiles.h), so that the gradient has that kernel's
// bits. Summed in one chain, q/k/v's at 1276 tokens is 8e-6 of its norm away, as close to the exact one
// (4.7e-4), and the training step's adapter gradients, 28 layers further, 4e-3. The slices' second set
// of accumulators costs 15.7 -> 16.4 us at 1276 tokens of 1536 -> 1536 + 256 + 256, 12.5 -> 14.0 at 65.
int dx_slices(int M, int K, int stages) {
  return K % 128 ? 1 : cm::nf4_tiles(M, K, K % 256 == 0, true, stages).split;
}

bool al16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

}  // namespace

extern "C" int cm_linear_f16_fwd(const void* x, int64_t ldx, int64_t M, int K, const void* w,
                                 int n_out, const int* N, const void* const* bias,
                                 void* const* out, const int64_t* ldo, void* stream) {
  CM_CHECK_ARG(M >= 0 && M < (int64_t{1} << 30) && K > 0 && K % 64 == 0);
  CM_CHECK_ARG(n_out >= 1 && n_out <= kMaxOut && N && out && ldo);
  Outputs o{};
  int64_t total = 0;
  for (int i = 0; i < kMaxOut; ++i) {
    o.first[i] = i < n_out ? static_cast<int>(total) : 0x7fffffff;
    if (i >= n_out) continue;
    CM_CHECK_ARG(N[i] > 0 && N[i] % 64 == 0 && N[i] <= (1 << 28));
    CM_CHECK_ARG(M == 0 || (out[i] && al16(out[i]) && ldo[i] >= N[i] && ldo[i] % 8 == 0));
    o.p[i] = static_cast<_Float16*>(out[i]);
    o.ld[i] = ldo[i];
    o.bias[i] = bias ? static_cast<const _Float16*>(bias[i]) : nullptr;
    total += N[i];
  }
  if (M == 0) return 0;
  CM_CHECK_ARG(x && w && al16(x) && al16(w) && ldx >= K && ldx % 8 == 0 && ldx < (1 << 22));
  CM_CHECK_ARG(K < (1 << 22) && total < (int64_t{1} << 30));
  const int m = static_cast<int>(M), n = static_cast<int>(total);
  const RowMajor a{static_cast<const _Float16*>(x), ldx, m, K};
  const RowMajor b{static_cast<const _Float16*>(w), K, n, K};
  hipStream_t s = static_cast<hipStream_t>(stream);
  return launch_best<false>(a, b, o, m, n, K, 1, s);
}

extern "C" int cm_linear_f16_bwd(const void* const* grad, const int64_t* ldg, int64_t M, int n_in,
                                 const int* N, const void* w, int K, void* dx, int64_t ldx,
                                 void* stream) {
  CM_CHECK_ARG(M >= 0 && M < (int64_t{1} << 30) && K > 0 && K % 64 == 0);
  CM_CHECK_ARG(n_in >= 1 && n_in <= kMaxOut && N && grad && ldg);
  SegRows g{};
  int64_t total = 0;
  for (int i = 0; i < kMaxOut; ++i) {
    g.first[i] = i < n_in ? static_cast<int>(total) : 0x7fffffff;
    if (i >= n_in) continue;
    CM_CHECK_ARG(N[i] > 0 && N[i] % 64 == 0 && N[i] <= (1 << 28));
    CM_CHECK_ARG(M == 0 || (grad[i] && al16(grad[i]) && ldg[i] >= N[i] && ldg[i] % 8 == 0 &&
                            ldg[i] < (1 << 22)));
    g.p[i] = static_cast<const _Float16*>(grad[i]);
    g.ld[i] = ldg[i];
    total += N[i];
  }
  if (M == 0) return 0;
  CM_CHECK_ARG(w && dx && al16(w) && al16(dx) && ldx >= K && ldx % 8 == 0);
  CM_CHECK_ARG(K < (1 << 22) && total < (int64_t{1} << 30));
  const int m = static_cast<int>(M), n = static_cast<int>(total);
  g.rows = m;
  g.k_len = n;
  const KMajor b{static_cast<const _Float16*>(w), K, K, n};
  Outputs o{};
  o.p[0] = static_cast<_Float16*>(dx);
  o.ld[0] = ldx;
  o.first[1] = o.first[2] = 0x7fffffff;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int slices = dx_slices(m, K, n / 64);
  return slices > 1 ? launch_best<true>(g, b, o, m, K, n, slices, s)
                    : launch_best<false>(g, b, o, m, K, n, 1, s);
}
