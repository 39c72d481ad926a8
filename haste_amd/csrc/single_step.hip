// One time step of an LSTM or GRU forward pass as one kernel: what ForwardPass::Iterate
// (reference lib/haste/lstm.h:73-86, lib/haste/gru.h:72-84) is called for in autoregressive
// decoding and streaming.  The all-steps kernels keep a slice of R on chip for a whole
// sequence; for a single step there is nothing to keep -- every weight is used once -- and
// their set-up (roles, exchange tiles, the slice, a group barrier) and the separate x * W
// launch cost more than the step.  Here [x_t | h] (length C + H) is multiplied with the stacked
// [W; R] straight from memory: a workgroup takes 16 hidden units (all their gate columns), 16 or
// 32 batch rows and a run of the contraction, parks its partial sums, and the last workgroup of
// an output tile to finish adds the runs in index order and does the pointwise step (gates, cell
// update, zoneout) -- one launch, no float atomics, results independent of timing.  The GRU's
// half entry points use the same kernel on half tensors (sums and pointwise step in float), and the
// double ones in double.
//
// Arithmetic: reference lib/lstm_forward_gpu.cu.cc:55-86, lib/gru_forward_gpu.cu.cc:46-84.
#include <algorithm>

#include "recurrent.h"

namespace haste_hip {
namespace {

constexpr int kStepUnits = 16;      // hidden units per workgroup
constexpr int kGroupRows = 16;      // contraction indices per group: four matrix instructions
constexpr int kBatchGroups = 4;     // groups whose weights a wavefront has in flight
constexpr int kStageGroups = 16;    // groups whose inputs are staged in LDS at a time
constexpr int kStageStride = kStageGroups * kGroupRows + 4;  // floats a row: 16-byte reads of 16 rows meet all banks
constexpr int kStepTiles = 4096;    // output tiles: the counters of the control block

typedef _Float16 half_t;
typedef double double4_t __attribute__((ext_vector_type(4)));

// What sums and the pointwise step are in, and the matrix instruction: A[row = lane % 16][k = lane / 16] times
// B[k = lane / 16][column = lane % 16]; element i of a lane is row row(lane, i) and column lane % 16.
template <typename T> struct Step {
  typedef float Sum;
  typedef float4_t Sum4;
  static constexpr bool kQuads = true;  // a lane's elements are rows of one quad
  static __device__ __forceinline__ Sum4 mfma(float a, float b, Sum4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int lane, int i) { return 4 * (lane >> 4) + i; }
  static __device__ __forceinline__ float sigmoid(float x) { return sigmoid_f(x); }
  static __device__ __forceinline__ float tanh_(float x) { return tanh_f(x); }
};
template <> struct Step<double> {
  typedef double Sum;
  typedef double4_t Sum4;
  static constexpr bool kQuads = false;
  static __device__ __forceinline__ Sum4 mfma(double a, double b, Sum4 c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int lane, int i) { return (lane >> 4) + 4 * i; }
  static __device__ __forceinline__ double sigmoid(double x) { return 1.0 / (1.0 + exp(-x)); }
  static __device__ __forceinline__ double tanh_(double x) { return tanh(x); }
};

// T: the caller's tensors (float, double, or half with the sums and the pointwise step in float).
template <typename T>
struct StepParams {
  int training, N, C, H;
  const T* W;            // [C, G*H]
  const T* R;            // [H, G*H]
  const T* b;            // LSTM: [4H]; GRU: bx [3H]
  const T* br;           // GRU: [3H]
  const T* x;            // [N, C]
  const T* h;            // [N, H]
  const T* c;            // LSTM: [N, H]
  T* h_out;              // [N, H]
  T* c_out;              // LSTM: [N, H]
  T* v;                  // [N, 4H] (training; GRU: always when non-null)
  float zoneout_prob;
  const T* zoneout_mask;      // [N, H] or null
  const T* dc_mask;           // DropConnect mask of R or null
  float dc_scale;
  typename Step<T>::Sum* h_stage;  // [N, H] where h_out is memory that others still read (StepStaging), else null
  typename Step<T>::Sum* c_stage;  // LSTM: the same for c_out
  int copies;                      // whether the kernel also copies them where they belong
  typename Step<T>::Sum* partial;  // [runs][output tiles][4 sums][quads of rows][64]; unused with one run
  ControlBlock* cb;
  int runs, row_blocks, unit_blocks, quads;  // quads: of rows, in an output tile
};

// Sums between workgroups of a launch (agent scope: store_agent, load_exchanged).
__device__ __forceinline__ float load_sum(const float* p) { return load_exchanged(p); }
__device__ __forceinline__ double load_sum(const double* p) {
  return __longlong_as_double((long long)__hip_atomic_load(reinterpret_cast<const unsigned long long*>(p), __ATOMIC_RELAXED,
                                                           __HIP_MEMORY_SCOPE_AGENT));
}
__device__ __forceinline__ void store_sum(float* p, float v) { store_agent(p, v); }
__device__ __forceinline__ void store_sum(double* p, double v) {
  __hip_atomic_store(reinterpret_cast<unsigned long long*>(p), (unsigned long long)__double_as_longlong(v),
                     __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void store_sum4(float* p, float4_t v) {
  unsigned long long* q = reinterpret_cast<unsigned long long*>(p);
  const unsigned long long lo = (unsigned long long)__float_as_uint(v.y) << 32 | __float_as_uint(v.x);
  const unsigned long long hi = (unsigned long long)__float_as_uint(v.w) << 32 | __float_as_uint(v.z);
  __hip_atomic_store(q, lo, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __hip_atomic_store(q + 1, hi, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void store_sum4(double* p, double4_t v) {
#pragma unroll
  for (int i = 0; i < 4; ++i) store_sum(p + i, v[i]);
}

// What the pointwise step of one unit of one row reads beside the sums.
template <typename A>
struct UnitInputs {
  A h, c, b[4], mask;
};

template <int GATES, typename T>
__device__ __forceinline__ UnitInputs<typename Step<T>::Sum> unit_inputs(const StepParams<T>& p, int n, int j) {
  typedef typename Step<T>::Sum A;
  UnitInputs<A> u = {};
  const int H = p.H;
  const size_t e = (size_t)n * H + j;
  u.h = (A)p.h[e];
  if constexpr (GATES == 4) {
    u.c = (A)p.c[e];
#pragma unroll
    for (int g = 0; g < 4; ++g) u.b[g] = (A)p.b[g * H + j];
  } else {
    u.b[0] = (A)p.b[j] + (A)p.br[j];
    u.b[1] = (A)p.b[H + j] + (A)p.br[H + j];
    u.b[2] = (A)p.b[2 * H + j];
    u.b[3] = (A)p.br[2 * H + j];
  }
  if (p.training && p.zoneout_prob != 0.f && p.zoneout_mask != nullptr) u.mask = (A)p.zoneout_mask[e];
  return u;
}

// Unit j of row n from its sums a: LSTM the four gates of [x | h] * [W; R]; GRU the update and the
// reset gate, x * W and h * R of the candidate gate.
template <int GATES, bool STAGED, typename T>
__device__ __forceinline__ void finish_unit(const StepParams<T>& p, int n, int j, const typename Step<T>::Sum (&a)[4],
                                            const UnitInputs<typename Step<T>::Sum>& in) {
  typedef typename Step<T>::Sum A;
  typedef Step<T> S;
  const int H = p.H;
  const size_t e = (size_t)n * H + j;
  const bool zoneout = p.zoneout_prob != 0.f && p.zoneout_mask != nullptr;
  A h_new;
  if constexpr (GATES == 4) {
    const A gi = S::sigmoid(a[0] + in.b[0]), gg = S::tanh_(a[1] + in.b[1]);
    const A gf = S::sigmoid(a[2] + in.b[2]), go = S::sigmoid(a[3] + in.b[3]);
    const A c_new = gf * in.c + gi * gg;
    h_new = go * S::tanh_(c_new);
    if (!STAGED || p.c_stage == nullptr) p.c_out[e] = (T)c_new;
    else store_sum(&p.c_stage[e], c_new);
    if (p.training) {
      T* vt = p.v + (size_t)n * 4 * H + j;
      vt[0] = (T)gi; vt[H] = (T)gg; vt[2 * H] = (T)gf; vt[3 * H] = (T)go;
    }
  } else {
    const A z = S::sigmoid(a[0] + in.b[0]);
    const A r = S::sigmoid(a[1] + in.b[1]);
    const A qg = a[3] + in.b[3];
    const A g = S::tanh_(a[2] + r * qg + in.b[2]);
    h_new = z * in.h + (A(1) - z) * g;
    if (p.training && p.v != nullptr) {
      T* vt = p.v + (size_t)n * 4 * H + j;
      vt[0] = (T)z; vt[H] = (T)r; vt[2 * H] = (T)g; vt[3 * H] = (T)qg;
    }
  }
  if (zoneout) {
    if (p.training) h_new = (h_new - in.h) * in.mask + in.h;
    else h_new = A(p.zoneout_prob) * in.h + (A(1) - A(p.zoneout_prob)) * h_new;
  }
  if (!STAGED || p.h_stage == nullptr) p.h_out[e] = (T)h_new;
  else store_sum(&p.h_stage[e], h_new);
}

// Elements first, first + stride .. of a parked state go where they belong, COPY of them on their way at a time.
template <int COPY, typename T>
__device__ __forceinline__ void copy_state(typename Step<T>::Sum* stage, T* out, int first, int stride, int count) {
  typedef typename Step<T>::Sum A;
  for (int i = first; i < count; i += COPY * stride) {
    A v[COPY];
#pragma unroll
    for (int k = 0; k < COPY; ++k) v[k] = i + k * stride < count ? load_sum(&stage[i + k * stride]) : A(0);
#pragma unroll
    for (int k = 0; k < COPY; ++k)
      if (i + k * stride < count) out[i + k * stride] = (T)v[k];
  }
}

// h_out or c_out overlaps h or x: other workgroups may still be reading them when a column block is
// finished, so the new state is parked.  Few elements (StepParams::copies) are copied out by the last column block to
// finish, when every run of every block has been read.  Called by the finishing workgroups, all threads.
template <typename T>
__device__ __forceinline__ void copy_staged_states(const StepParams<T>& p, unsigned int* flag) {
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (threadIdx.x == 0) {
    const unsigned int old = __hip_atomic_fetch_add(&p.cb->grid_exit_counter[0], 1u, __ATOMIC_RELAXED,
                                                    __HIP_MEMORY_SCOPE_AGENT);
    const bool last = old == (unsigned)(p.row_blocks * p.unit_blocks) - 1u;
    if (last)
      __hip_atomic_store(&p.cb->grid_exit_counter[0], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    *flag = last ? 1u : 0u;
  }
  __syncthreads();
  if (*flag == 0u) return;
  const int count = p.N * p.H;
  if (p.h_stage != nullptr) copy_state<4, T>(p.h_stage, p.h_out, threadIdx.x, 256, count);
  if (p.c_stage != nullptr) copy_state<4, T>(p.c_stage, p.c_out, threadIdx.x, 256, count);
}

// More of them: a launch of its own.
template <typename T>
__global__ __launch_bounds__(256)
void copy_staged_kernel(typename Step<T>::Sum* h_stage, T* h_out, typename Step<T>::Sum* c_stage, T* c_out, int count) {
  const int first = blockIdx.x * 256 + threadIdx.x, stride = gridDim.x * 256;
  if (h_stage != nullptr) copy_state<4, T>(h_stage, h_out, first, stride, count);
  if (c_stage != nullptr) copy_state<4, T>(c_stage, c_out, first, stride, count);
}

// GATES = 4: LSTM (i, g, f, o); GATES = 3: GRU (z, r, g).  RT: tiles of 16 batch rows a workgroup
// takes.  [W; R] in groups of 16 rows, each side's last group filled up with zeros; a workgroup
// takes run `run` of the groups.  Wavefront w sums gate w of its 16 units; for the GRU's
// candidate gate, whose two sides meet the reset gate apart, wavefront 2 takes W and wavefront 3 R.
// Every weight goes from memory to the register of the one lane that feeds it to the matrix unit
// (fp32 instruction: 16 rows of a batch against 16 units cost a quarter of what the loads take);
// the inputs are staged in LDS.  Lane (column l % 16, l / 16) of a group's i-th instruction holds
// contraction index 4 (l / 16) + i, so that its inputs are one 16-byte read.  STAGED: some of the new state is parked.
template <int GATES, int RT, bool DROPCONNECT, bool STAGED, typename T>
__global__ __launch_bounds__(256)
void forward_step_kernel(StepParams<T> p) {
  typedef typename Step<T>::Sum A;
  typedef typename Step<T>::Sum4 A4;
  __shared__ __attribute__((aligned(16))) A s_in[RT * 16 * kStageStride];
  __shared__ unsigned int s_flag;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int N = p.N, H = p.H;
  // Workgroups go to the XCDs in turn: each XCD is given a range of the work, the row blocks and
  // then the column blocks that share weights (and halves of 128-byte lines of them) side by side.
  const int total = gridDim.x, xcd = blockIdx.x & 7, each = total >> 3, rest = total & 7;
  const int work = xcd * each + (xcd < rest ? xcd : rest) + (blockIdx.x >> 3);
  const int tiles = p.row_blocks * p.unit_blocks;
  const int run = work / tiles, tile = work % tiles;
  const int rb = tile % p.row_blocks, cw = tile / p.row_blocks;
  const int n0 = rb * RT * 16, j0 = cw * kStepUnits;

  const int len_w = p.C, len_r = H;
  const int groups_w = (len_w + kGroupRows - 1) / kGroupRows;
  const int groups = groups_w + (len_r + kGroupRows - 1) / kGroupRows;
  const int first = (int)((long long)run * groups / p.runs), last = (int)((long long)(run + 1) * groups / p.runs);
  // this wavefront's groups
  const int my_first = GATES == 3 && wave == 3 && first < groups_w ? groups_w : first;
  const int my_last = GATES == 3 && wave == 2 && last > groups_w ? groups_w : last;
  const int gate = GATES == 3 && wave == 3 ? 2 : wave;
  const int unit = j0 + (lane & 15) < H ? j0 + (lane & 15) : H - 1;  // columns beyond H are computed and dropped
  const int k_lane = 4 * (lane >> 4);
  const unsigned row_bytes = (unsigned)GATES * H * sizeof(T), column = ((unsigned)gate * H + unit) * sizeof(T);
  const char *const W = reinterpret_cast<const char*>(p.W), *const R = reinterpret_cast<const char*>(p.R);

  // The weights of kBatchGroups groups from group g on.  Nothing is read outside W and R: rows beyond a
  // side's end are read from its last row, groups beyond the run from its last group (neither is used).
  auto load_weights = [&](int g, T (&w)[kBatchGroups][4], T (&m)[kBatchGroups][4]) {
#pragma unroll
    for (int q = 0; q < kBatchGroups; ++q) {
      const int gg = g + q < last ? g + q : last - 1;
      const bool recurrent = gg >= groups_w;
      const int k0 = (recurrent ? gg - groups_w : gg) * kGroupRows, left = (recurrent ? len_r : len_w) - k0;
      const char* M = (recurrent ? R : W) + (size_t)k0 * row_bytes;
      const unsigned end = (unsigned)(left - 1) * row_bytes + column;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const unsigned full = (unsigned)(k_lane + i) * row_bytes + column;
        const unsigned at = left >= kGroupRows || full < end ? full : end;
        w[q][i] = *reinterpret_cast<const T*>(M + at);
        if constexpr (DROPCONNECT) {
          // (for W: any value, not used)
          const char* mask = reinterpret_cast<const char*>(p.dc_mask) + (recurrent ? (size_t)k0 * row_bytes : 0);
          m[q][i] = *reinterpret_cast<const T*>(mask + (recurrent ? at : column));
        }
      }
    }
  };

  const A4 zero4 = {A(0), A(0), A(0), A(0)};
  A4 acc[RT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) acc[rt] = zero4;
  // Groups g .., staged from s0 on.  Every batch is summed by itself, in four sums side by side: short chains,
  // whose rounding errors stay those of many small runs.
  auto multiply = [&](int g, int s0, const T (&w)[kBatchGroups][4], const T (&m)[kBatchGroups][4]) {
    A4 part[RT][4];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int i = 0; i < 4; ++i) part[rt][i] = zero4;
#pragma unroll
    for (int q = 0; q < kBatchGroups; ++q) {
      const int gg = g + q;
      if (gg < my_first || gg >= my_last) continue;  // the same for a whole wavefront
      const bool recurrent = gg >= groups_w;
      const int left = (recurrent ? len_r : len_w) - (recurrent ? gg - groups_w : gg) * kGroupRows;
      A4 a[RT];
#pragma unroll
      for (int rt = 0; rt < RT; ++rt)
        a[rt] = *reinterpret_cast<const A4*>(
            &s_in[(rt * 16 + (lane & 15)) * kStageStride + (gg - s0) * kGroupRows + k_lane]);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        A weight = (A)w[q][i];
        if constexpr (DROPCONNECT) weight = recurrent ? weight * (A)m[q][i] * A(p.dc_scale) : weight;
        weight = k_lane + i < left ? weight : A(0);
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
          part[rt][i] = Step<T>::mfma(a[rt][i], weight, part[rt][i]);
      }
    }
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) acc[rt] += (part[rt][0] + part[rt][1]) + (part[rt][2] + part[rt][3]);
  };
  // The inputs of groups s0 ..: lane l takes contraction index l of 64, a wavefront every fourth row.
  auto stage = [&](int s0) {
    if (s0 != first) __syncthreads();
    const int s1 = s0 + kStageGroups < last ? s0 + kStageGroups : last;
    for (int g = s0; g < s1; g += 4) {
      const int mine = g + (lane >> 4) < last ? g + (lane >> 4) : last - 1;
      const bool recurrent = mine >= groups_w;
      const int len = recurrent ? len_r : len_w, k = (recurrent ? mine - groups_w : mine) * kGroupRows + (lane & 15);
      const T* in = (recurrent ? p.h : p.x) + (k < len ? k : len - 1);
      A value[4 * RT];
#pragma unroll
      for (int i = 0; i < 4 * RT; ++i) {
        const int n = n0 + wave + 4 * i;
        value[i] = (A)in[(size_t)(n < N ? n : N - 1) * len];
      }
#pragma unroll
      for (int i = 0; i < 4 * RT; ++i)
        s_in[(wave + 4 * i) * kStageStride + (g - s0) * kGroupRows + lane] =
            k < len && n0 + wave + 4 * i < N ? value[i] : A(0);
    }
    __syncthreads();
  };
  // Two batches of weights in turn: one is used while the next is on its way.
  T w0[kBatchGroups][4], w1[kBatchGroups][4], m0[kBatchGroups][4], m1[kBatchGroups][4];
  load_weights(first, w0, m0);
  int s0 = first;
  stage(s0);
  if (first + kBatchGroups < last) load_weights(first + kBatchGroups, w1, m1);
  multiply(first, s0, w0, m0);
  for (int g = first + kBatchGroups; g < last;) {
    load_weights(g + kBatchGroups, w0, m0);
    if (g == s0 + kStageGroups) stage(s0 = g);
    multiply(g, s0, w1, m1);
    g += kBatchGroups;
    if (g >= last) break;
    load_weights(g + kBatchGroups, w1, m1);
    if (g == s0 + kStageGroups) stage(s0 = g);
    multiply(g, s0, w0, m0);
    g += kBatchGroups;
  }

  // Lane l of wavefront w holds sum w of four rows of each tile and unit l % 16.  Thread t finishes element t % 4
  // of lane t / 4: its sums lie side by side with its neighbours'.
  const int row = Step<T>::row(tid >> 2, tid & 3), j = j0 + ((tid >> 2) & 15);
  const unsigned slot = 64 * p.quads, run_stride = tiles * 4 * slot;  // one sum of a tile, all of a run
  if (p.runs == 1) {
    __syncthreads();
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
      *reinterpret_cast<A4*>(&s_in[(wave * RT + rt) * 256 + 4 * lane]) = acc[rt];
  } else {
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
      if (!Step<T>::kQuads || 4 * rt + (lane >> 4) < p.quads)
        store_sum4(p.partial + run * run_stride + (4 * tile + wave) * slot + rt * 256 + 4 * lane, acc[rt]);
  }
  // What the pointwise step reads is on its way while the sums are handed over.
  UnitInputs<A> in[RT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    in[rt] = UnitInputs<A>{};
    const int n = n0 + 16 * rt + row;
    if (n < N && j < H) in[rt] = unit_inputs<GATES, T>(p, n, j);
  }
  if (p.runs == 1) __syncthreads();
  else if (!column_last_arrival(p.cb, tile, p.runs, &s_flag)) return;
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    const int n = n0 + 16 * rt + row;
    if (n >= N || j >= H) continue;
    A a[4] = {A(0), A(0), A(0), A(0)};
    if (p.runs == 1) {
#pragma unroll
      for (int g = 0; g < 4; ++g) a[g] = s_in[(g * RT + rt) * 256 + tid];
    } else {
      const unsigned at = 4 * tile * slot + rt * 256 + tid;
      for (int r0 = 0; r0 < p.runs; r0 += 16) {  // 64 loads in flight
        A run_sum[16][4];
#pragma unroll
        for (int i = 0; i < 16; ++i)
#pragma unroll
          for (int g = 0; g < 4; ++g)
            run_sum[i][g] = r0 + i < p.runs ? load_sum(p.partial + (at + (r0 + i) * run_stride + g * slot)) : A(0);
#pragma unroll
        for (int width = 8; width > 0; width /= 2)
#pragma unroll
          for (int i = 0; i < width; ++i)
#pragma unroll
            for (int g = 0; g < 4; ++g) run_sum[i][g] += run_sum[i + width][g];
#pragma unroll
        for (int g = 0; g < 4; ++g) a[g] += run_sum[0][g];
      }
    }
    finish_unit<GATES, STAGED, T>(p, n, j, a, in[rt]);
  }
  if (STAGED && p.copies) copy_staged_states(p, &s_flag);
}

// How a step is cut up.
struct StepCut {
  int rt, row_blocks, unit_blocks, runs, quads;
  size_t sums() const {
    return runs > 1 ? (size_t)runs * row_blocks * unit_blocks * 4 * 64 * quads : 0;
  }
};

// Blocks of 16 units, 16 rows and 16 contraction indices.
long long step_blocks(int N, int C, int H) {
  const long long groups = (C + kGroupRows - 1) / kGroupRows + (H + kGroupRows - 1) / kGroupRows;
  return (long long)((N + 15) / 16) * ((H + kStepUnits - 1) / kStepUnits) * groups;
}

// A step is bound by the latency of its chain (loads, sums out, a counter, sums in).
// Up to 16 rows a run is as few batches of weights (kBatchGroups groups, which are on their way together: a run of a batch
// and a group takes two) as leave no more workgroups than a CU holds well at a time (three, with runs of more than 16
// batches four, in double two) and not many more runs than batches: every run's sums meet in memory.  Measured, N = 1,
// us by batches a run:
//   float   C =  64, H =  256  1: 6.4   2: 7.3   3: 8.1   5 (one run): 8.5
//           C =  64, H =  512  1: 7.6   2: 7.9   3: 8.5   5: 10.6
//           C = 512, H =  512  1: 9.4   2: 8.7   4: 9.3
//           C = 256, H = 1024  1: 12.8  2: 10.9  3: 11.6  4: 12.3
//           C =  64, H = 2048  1: 25.4  3: 20.1  4: 20.5  6: 20.8  9: 21.2
//   double  C =  64, H =  512  1: 11.7  2: 11.1  3: 12.1
//           C = 512, H = 1536  2: 45.6  4: 32.6  8: 33.6
// With more rows, runs of at least 8 groups, whose sums are then read by fewer: two workgroups per CU (double at most two:
// N = 24, C = 64, H = 1280, 480 / 560 workgroups 25 / 38; float three: N = 320, C = 64, H = 768, 480 / 960 32 / 43), in float and
// half, where that leaves runs of more than 32 groups, up to four.
// 32 rows a workgroup halve the reading of weights, once there are enough tiles for it (LSTM,
// C = H = 512, us with 16 / 32 rows: N = 64, 128 tiles of 16, 12.2 / 14.2; N = 128, 256 tiles, 17.6 / 16.5).
StepCut step_cut(int N, int C, int H, size_t element) {
  StepCut s;
  const int cus = device_cu_count() > 0 ? device_cu_count() : 256;
  s.unit_blocks = (H + kStepUnits - 1) / kStepUnits;
  s.rt = element < 8 && N > 16 && (N + 15) / 16 * (long long)s.unit_blocks >= cus ? 2 : 1;
  s.row_blocks = (N + 16 * s.rt - 1) / (16 * s.rt);
  s.quads = s.row_blocks > 1 || element == 8 ? 4 * s.rt : (N + 3) / 4;
  const int groups = (C + kGroupRows - 1) / kGroupRows + (H + kGroupRows - 1) / kGroupRows;
  const long long tiles = (long long)s.row_blocks * s.unit_blocks;
  long long runs;
  if (s.rt == 1 && s.row_blocks == 1) {
    auto of = [&](int batches) { return (groups + batches * kBatchGroups - 1) / (batches * kBatchGroups); };
    auto fewest = [&](int per_cu) {
      int batches = groups <= 2 * kBatchGroups ? 2 : 1;
      while (of(batches) > 1 && (tiles * of(batches) > (long long)per_cu * cus || of(batches) > 10 * batches)) ++batches;
      return batches;
    };
    int batches = fewest(element == 8 ? 2 : 3);
    if (batches > 16 && element < 8) batches = fewest(4);
    runs = of(batches);
  } else if (element == 8) {
    runs = std::min<long long>(2 * cus / tiles, groups / 8);
  } else {
    runs = std::min<long long>((2 * cus + tiles - 1) / tiles, groups / 8);
    if (element == 4 && tiles * runs > 3 * cus) runs = 3 * cus / tiles;
    if (runs < groups / 32) runs = std::min<long long>((4 * cus + tiles - 1) / tiles, groups / 32);
  }
  s.runs = runs < 1 ? 1 : (int)runs;
  return s;
}

// Which results of a step are parked until all of its workgroups have read their inputs.  Every workgroup of a row block
// reads x and h; an element of c and of the mask only the thread that writes the results of that element.
struct StepStaging {
  bool h = false, c = false;
  bool possible = true;  // v is not parked
  size_t bytes = 0;
};

StepStaging step_staging(int N, int C, int H, size_t element, const StepTensors& t) {
  const size_t state = (size_t)N * H;
  auto overlaps = [&](const void* out, size_t out_count, const void* in, size_t in_count) {
    const uintptr_t to = reinterpret_cast<uintptr_t>(out), from = reinterpret_cast<uintptr_t>(in);
    return out != nullptr && in != nullptr && to < from + in_count * element && from < to + out_count * element;
  };
  auto read_by_others = [&](const void* out, size_t count) {
    return overlaps(out, count, t.x, (size_t)N * C) || overlaps(out, count, t.h, state) ||
           (overlaps(out, count, t.c, state) && out != t.c) || (overlaps(out, count, t.mask, state) && out != t.mask);
  };
  StepStaging s;
  if (planned_pass() != nullptr) return s;  // (whose tensors are all at one address)
  s.h = read_by_others(t.h_out, state);
  s.c = read_by_others(t.c_out, state);
  s.possible = !read_by_others(t.v, 4 * state) && (t.v == nullptr || (t.v != t.c && t.v != t.mask));
  s.bytes = ((s.h ? 1 : 0) + (s.c ? 1 : 0)) * state * (element == 8 ? 8 : 4);
  return s;
}

// Elements of parked states up to which the step's last workgroup copies them, a memory round trip for every 1024; a launch
// of its own costs 2 - 3 us at any size.  (A step in place of N x H, C = 64, us in the step / with the launch: LSTM 4 x 64
// 6.3 / 8.1, 2 x 1024 12.3 / 13.1, 8 x 512 11.5 / 11.6, 16 x 512 13.2 / 11.8; half GRU 1 x 512 10.6 / 11.2, 4 x 512 12.1 / 11.6, 8 x 512
// 13.5 / 11.4; double LSTM 8 x 64 8.6 / 10.2, 8 x 256 13.1 / 13.6, 8 x 1024 21.2 / 19.2.)
constexpr size_t kCopiedInStep = 2048;

template <int GATES, typename T>
int launch_step(hipStream_t stream, StepParams<T>& p, const char* name) {
  typedef typename Step<T>::Sum A;
  StepCut cut = step_cut(p.N, p.C, p.H, sizeof(T));
  const StepStaging staging = step_staging(p.N, p.C, p.H, sizeof(T), {p.x, p.h, p.c, p.zoneout_mask, p.h_out, p.c_out,
                                                                      p.training ? p.v : nullptr});
  const size_t state_bytes = staging.bytes;
  for (bool room = false; !room && cut.runs > 1;) {
    HASTE_HIP_PROPAGATE(workspace_has_room(stream, cut.sums() * sizeof(A) + state_bytes + 256, &room));
    if (!room) cut.runs = (cut.runs + 1) / 2;
  }
  const size_t partial_bytes = cut.sums() * sizeof(A);
  Workspace ws;
  HASTE_HIP_PROPAGATE(get_workspace(stream, partial_bytes + state_bytes + 256, &ws));
  if (PlannedPass* pass = planned_pass()) {
    pass->kernel = kPlanSingleStep;
    return HASTE_HIP_OK;
  }
  p.partial = reinterpret_cast<A*>(ws.scratch);
  A* stage = p.partial + cut.sums();
  p.h_stage = staging.h ? stage : nullptr;
  p.c_stage = staging.c ? stage + (staging.h ? (size_t)p.N * p.H : 0) : nullptr;
  const size_t parked = state_bytes / sizeof(A);
  p.copies = parked > 0 && parked <= kCopiedInStep;
  p.cb = ws.control;
  p.runs = cut.runs; p.row_blocks = cut.row_blocks; p.unit_blocks = cut.unit_blocks; p.quads = cut.quads;
  const dim3 grid((unsigned)cut.row_blocks * cut.unit_blocks * cut.runs);
  ScopedKernelTimer timer(name, stream);
#define HASTE_LAUNCH_STEP(RT_)                                                                                     \
  if (cut.rt == RT_) {                                                                                             \
    if (p.dc_mask != nullptr && parked) forward_step_kernel<GATES, RT_, true, true, T><<<grid, 256, 0, stream>>>(p); \
    else if (p.dc_mask != nullptr) forward_step_kernel<GATES, RT_, true, false, T><<<grid, 256, 0, stream>>>(p);     \
    else if (parked) forward_step_kernel<GATES, RT_, false, true, T><<<grid, 256, 0, stream>>>(p);                   \
    else forward_step_kernel<GATES, RT_, false, false, T><<<grid, 256, 0, stream>>>(p);                              \
  }
  HASTE_LAUNCH_STEP(1)
  if constexpr (Step<T>::kQuads) {
    HASTE_LAUNCH_STEP(2)
  }
#undef HASTE_LAUNCH_STEP
  HASTE_HIP_TRY(hipGetLastError());
  if (parked > kCopiedInStep) {
    const unsigned count = (unsigned)p.N * p.H;
    copy_staged_kernel<T><<<dim3((count + 1023) / 1024), dim3(256), 0, stream>>>(p.h_stage, p.h_out, p.c_stage, p.c_out, (int)count);
    HASTE_HIP_TRY(hipGetLastError());
  }
  return HASTE_HIP_OK;
}

}  // namespace

// Whether a step of N rows is this kernel's rather than what it would run on otherwise.  In float and half up to 8 rows
// always, as long as its tiles have counters.  Beyond (blocks: of 16 units, rows and contraction indices; tiles: of 16 or 32
// rows, which up to one per CU do not wait for one another; us there / here):
//  - float, all-steps kernels, which fetch their slice of R for one use: N = 43, C = 32, H = 128 13.6 / 5.7; N = 64, C = 64,
//    H = 2048 82 / 55; N = 256, C = 512, H = 1024 (98 304 blocks) 66 / 51.
//  - float, a GEMM per side, which keeps more of both operands on chip.  Up to H = 1024 slower as long as there are few
//    blocks: N = 160, C = 64, H = 768 33 / 22, N = 160, C = 512, H = 1024 (61 440, 320 tiles) 48 / 42, N = 512, C = 512, H = 448
//    (53 760, 448 tiles) 47 / 37; but with many tiles of a long contraction N = 208, C = 64, H = 1024 (56 576, 448 tiles) 40 / 51,
//    and N = 320, C = 64, H = 896 (67 200) 38 / 47.  Beyond, with tiles for every CU at most: N = 96, C = 64, H = 1280 (240 tiles) 34 / 29, GRU 31 / 29; but
//    N = 112, H = 1152 (288) 33 / 37 and N = 80, H = 1536 (288) 39 / 45.  From where no batch has a resident slice, the GEMM's
//    small form: N = 16, C = 64, H = 2560 27 / 31, GRU 24 / 27; N = 16, H = 4096 52 / 60.
//  - half, where the other way converts its weights: N = 64, C = 64, H = 2048 127 / 42, N = 128, C = 512, H = 4096 420 / 238.
//  - double, a product per side and a pointwise launch: LSTM N = 1, C = H = 512 17.4 / 11.1, GRU N = 8, C = 512, H = 1536
//    (12 288) 31 / 25, N = 128, C = H = 512 (16 384, 256 tiles) 33 / 28; more tiles than CUs N = 320, C = 64, H = 256 (6 400)
//    22 / 17, but N = 128, C = 64, H = 576 (11 520, 288 tiles) 25 / 28.
static bool step_pays(StepOther other, long long blocks, long long tiles, int H) {
  const int cus = device_cu_count() > 0 ? device_cu_count() : 256;
  switch (other) {
    case kStepResident: return blocks <= 128 << 10;
    case kStepStreamed:
      if (H > 1024) return blocks <= 60 << 10 && H <= 2048 && tiles <= cus;
      return blocks <= (2 * tiles <= 3 * cus || H <= 512 ? 60 << 10 : 48 << 10);
    case kStepHalf: return true;
    case kStepDouble: return blocks <= (tiles <= cus ? 16 << 10 : 8 << 10);
  }
  return false;
}

int single_step_rule(hipStream_t stream, int N, int C, int H, size_t element, StepOther other, const StepTensors& tensors,
                     bool* applies) {
  const StepCut cut = step_cut(N, C, H, element);
  const StepStaging staging = step_staging(N, C, H, element, tensors);
  const long long tiles = (long long)cut.row_blocks * cut.unit_blocks;
  *applies = tiles <= kStepTiles && staging.possible;
  if (!*applies || (N <= 8 && element != 8)) return HASTE_HIP_OK;
  *applies = step_pays(other, step_blocks(N, C, H), tiles, H);
  if (!*applies) return HASTE_HIP_OK;
  return workspace_has_room(stream, cut.sums() * (element == 8 ? 8 : 4) + staging.bytes + 256, applies);
}

int lstm_forward_single_step(hipStream_t stream, int training, int N, int C, int H, const float* W,
                             const float* R, const float* b, const float* x, const float* h,
                             const float* c, float* h_out, float* c_out, float* v,
                             float zoneout_prob, const float* zoneout_mask, const float* dc_mask,
                             float dc_scale) {
  StepParams<float> p = {};
  p.training = training; p.N = N; p.C = C; p.H = H;
  p.W = W; p.R = R; p.b = b; p.x = x; p.h = h; p.c = c;
  p.h_out = h_out; p.c_out = c_out; p.v = v;
  p.zoneout_prob = zoneout_prob; p.zoneout_mask = zoneout_mask;
  p.dc_mask = dc_mask; p.dc_scale = dc_scale;
  return launch_step<4>(stream, p, "lstm_forward_step");
}

int gru_forward_single_step(hipStream_t stream, int training, int N, int C, int H, const float* W,
                            const float* R, const float* bx, const float* br, const float* x,
                            const float* h, float* h_out, float* v, float zoneout_prob,
                            const float* zoneout_mask, const float* dc_mask, float dc_scale) {
  StepParams<float> p = {};
  p.training = training; p.N = N; p.C = C; p.H = H;
  p.W = W; p.R = R; p.b = bx; p.br = br; p.x = x; p.h = h;
  p.h_out = h_out; p.v = v;
  p.zoneout_prob = zoneout_prob; p.zoneout_mask = zoneout_mask;
  p.dc_mask = dc_mask; p.dc_scale = dc_scale;
  return launch_step<3>(stream, p, "gru_forward_step");
}

int lstm_forward_single_step(hipStream_t stream, int training, int N, int C, int H, const double* W,
                             const double* R, const double* b, const double* x, const double* h,
                             const double* c, double* h_out, double* c_out, double* v,
                             float zoneout_prob, const double* zoneout_mask, const double* dc_mask,
                             float dc_scale) {
  StepParams<double> p = {};
  p.training = training; p.N = N; p.C = C; p.H = H;
  p.W = W; p.R = R; p.b = b; p.x = x; p.h = h; p.c = c;
  p.h_out = h_out; p.c_out = c_out; p.v = v;
  p.zoneout_prob = zoneout_prob; p.zoneout_mask = zoneout_mask;
  p.dc_mask = dc_mask; p.dc_scale = dc_scale;
  return launch_step<4>(stream, p, "lstm_forward_step_double");
}

int gru_forward_single_step(hipStream_t stream, int training, int N, int C, int H, const double* W,
                            const double* R, const double* bx, const double* br, const double* x,
                            const double* h, double* h_out, double* v, float zoneout_prob,
                            const double* zoneout_mask, const double* dc_mask, float dc_scale) {
  StepParams<double> p = {};
  p.training = training; p.N = N; p.C = C; p.H = H;
  p.W = W; p.R = R; p.b = bx; p.br = br; p.x = x; p.h = h;
  p.h_out = h_out; p.v = v;
  p.zoneout_prob = zoneout_prob; p.zoneout_mask = zoneout_mask;
  p.dc_mask = dc_mask; p.dc_scale = dc_scale;
  return launch_step<3>(stream, p, "gru_forward_step_double");
}

int gru_forward_single_step_half(hipStream_t stream, int training, int N, int C, int H, const void* W,
                                 const void* R, const void* bx, const void* br, const void* x,
                                 const void* h, void* h_out, void* v, float zoneout_prob,
                                 const void* zoneout_mask, const void* dc_mask, float dc_scale) {
  auto in = [](const void* q) { return static_cast<const half_t*>(q); };
  StepParams<half_t> p = {};
  p.training = training; p.N = N; p.C = C; p.H = H;
  p.W = in(W); p.R = in(R); p.b = in(bx); p.br = in(br); p.x = in(x); p.h = in(h);
  p.h_out = static_cast<half_t*>(h_out); p.v = static_cast<half_t*>(v);
  p.zoneout_prob = zoneout_prob; p.zoneout_mask = in(zoneout_mask);
  p.dc_mask = in(dc_mask); p.dc_scale = dc_scale;
  return launch_step<3>(stream, p, "gru_forward_step_half");
}

}  // namespace haste_hip
