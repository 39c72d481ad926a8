// The states of a batch whose sequences have lengths of their own: what the layers return of a
// state sequence [T+1,N,H], and the way back.  (The reference's layers index their output with the
// lengths, frameworks/pytorch/base_rnn.py:54-61.)
//
// Bound: launches.  Indexing two sequences takes three launches of a tensor library (the batch indices, a
// gather each: 15 us for LSTM states of 16 x 256), its gradient six (zeros, a copy of the steps'
// gradients, indices, gather, sum, scatter: 24 us at T = 83, N = 37, H = 300); one each here, 3 and
// 6 us.  Only rows of the batch are gathered, and the gradient reads and writes every element once.
#include "common.h"

namespace haste_hip {
namespace {

constexpr int kStateThreads = 256;
// A launch has fewer than 2^32 threads: more rows than this are looped over.
constexpr int kMaxStateBlocks = 1 << 20;

// Step of the sequence [T+1,...] a length means: counted from the end when negative, -1 when there
// is no such step.
__device__ __forceinline__ long long step_of(long long length, int T) {
  const long long s = length < 0 ? length + T + 1 : length;
  return s < 0 || s > T ? -1 : s;
}

template <typename V>
struct StateJobs { const V* seq[2]; V* out[2]; };

// blockIdx.x: batch row (and those a grid further on), blockIdx.y: sequence.
template <typename V>
__global__ __launch_bounds__(kStateThreads)
void gather_states_kernel(int T, int N, int H, StateJobs<V> jobs, const long long* __restrict__ lengths) {
  for (unsigned n = blockIdx.x; n < (unsigned)N; n += gridDim.x) {
    const long long s = step_of(lengths[n], T);
    const V* from = jobs.seq[blockIdx.y] + ((size_t)(s < 0 ? 0 : s) * N + n) * H;
    V* to = jobs.out[blockIdx.y] + (size_t)n * H;
    for (int j = threadIdx.x; j < H; j += kStateThreads) to[j] = s < 0 ? V(__builtin_nanf("")) : from[j];
  }
}

// out[t][n] = grad[t][n] (0 without grad) + last[n] where t + 1 is the row's length; length 0 names
// the initial state, which is no step's.  A row whose length names no step had NaNs for a state: so are
// its gradients.
template <typename V>
__global__ __launch_bounds__(kStateThreads)
void state_gradients_kernel(int T, int N, int H, const V* __restrict__ grad, size_t step_stride, size_t row_stride,
                            const V* __restrict__ last, const long long* __restrict__ lengths, V* __restrict__ out) {
  for (unsigned row = blockIdx.x; row < (unsigned)T * (unsigned)N; row += gridDim.x) {
    const int t = row / (unsigned)N, n = row % (unsigned)N;
    const long long s = step_of(lengths[n], T);
    const V* from = grad + t * step_stride + n * row_stride;
    for (int j = threadIdx.x; j < H; j += kStateThreads) {
      V v = grad != nullptr ? from[j] : V(0);
      if (s == t + 1) v = v + last[(size_t)n * H + j];
      if (s < 0) v = V(__builtin_nanf(""));
      out[(size_t)row * H + j] = v;
    }
  }
}

unsigned state_blocks(long long rows) { return (unsigned)(rows < kMaxStateBlocks ? rows : kMaxStateBlocks); }

template <typename V>
int gather_states(int T, int N, int H, const V* seq0, const V* seq1, const void* lengths, V* out0, V* out1, void* stream) {
  HASTE_HIP_REQUIRE(T > 0 && N > 0 && H > 0 && seq0 && out0 && lengths && (seq1 == nullptr) == (out1 == nullptr));
  const StateJobs<V> jobs = {{seq0, seq1}, {out0, out1}};
  gather_states_kernel<V><<<dim3(state_blocks(N), seq1 != nullptr ? 2u : 1u), dim3(kStateThreads), 0, as_stream(stream)>>>(
      T, N, H, jobs, static_cast<const long long*>(lengths));
  HASTE_HIP_TRY(hipGetLastError());
  return HASTE_HIP_OK;
}

template <typename V>
int state_gradients(int T, int N, int H, const V* grad, size_t step_stride, size_t row_stride, const V* last,
                    const void* lengths, V* out, void* stream) {
  HASTE_HIP_REQUIRE(T > 0 && N > 0 && H > 0 && last && lengths && out && (long long)T * N < (1ll << 31));
  state_gradients_kernel<V><<<dim3(state_blocks((long long)T * N)), dim3(kStateThreads), 0, as_stream(stream)>>>(
      T, N, H, grad, step_stride, row_stride, last, static_cast<const long long*>(lengths), out);
  HASTE_HIP_TRY(hipGetLastError());
  return HASTE_HIP_OK;
}

}  // namespace
}  // namespace haste_hip

#define HASTE_STATES(SUFFIX, PUBLIC, V)                                                                              \
  extern "C" int haste_hip_gather_states_##SUFFIX(int T, int N, int H, const PUBLIC* seq0, const PUBLIC* seq1,       \
                                                  const void* lengths, PUBLIC* out0, PUBLIC* out1, void* stream) {   \
    return haste_hip::gather_states<V>(T, N, H, (const V*)seq0, (const V*)seq1, lengths, (V*)out0, (V*)out1, stream); \
  }                                                                                                                  \
  extern "C" int haste_hip_state_gradients_##SUFFIX(int T, int N, int H, const PUBLIC* grad, size_t step_stride,     \
                                                    size_t row_stride, const PUBLIC* last, const void* lengths,      \
                                                    PUBLIC* out, void* stream) {                                     \
    return haste_hip::state_gradients<V>(T, N, H, (const V*)grad, step_stride, row_stride, (const V*)last, lengths,  \
                                         (V*)out, stream);                                                           \
  }
HASTE_STATES(f32, float, float)
HASTE_STATES(f64, double, double)
HASTE_STATES(f16, void, _Float16)
#undef HASTE_STATES
