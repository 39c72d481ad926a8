// The recurrences of the LSTM and the GRU in double precision, all steps in one launch.
//
// Step-wise (stepwise.hip) a step is two launches, the product and the pointwise kernel, and
// most of its time is theirs: at N = 64, H = 512 the pair takes 15 us, and 9.3 us are left when
// its product loads no operand at all; the fp64 matrix cores need 1.7 us.  Here a workgroup keeps
// its columns of the weights in registers for the whole launch, and what the steps exchange goes
// through tiles in memory, behind the group's step barrier or polled (polled64).
//   * A group is 8 or 16 batch rows; its workgroups own HS hidden units each.  Forward: all gates of 8 or 16 units, the
//     contraction runs over h.  Backward: 16 units of dh, the contraction over all gate gradients.
//   * 16 rows: v_mfma_f64_16x16x4_f64.  8 rows: twice v_mfma_f64_4x4x4_4b_f64, four blocks of 4 x 4 at the same rate
//     (16.7 cycles for 512 flops, 70 for 2048), so that twice the groups share the work and 64 rows fill the eight
//     XCDs with a group each.  Forward the blocks are 16 columns and read the same A; backward, where A is the larger
//     part, they are 16 k, and the blocks' sums are added once a step.
//   * The four wavefronts take a quarter of the contraction each: at most KS instructions of four k,
//     a lane holding B[k = lane / 16][column = lane % 16] of every one of them and column tile.
//   * Exchange tile: what a lane needs next lies in one 16-byte word (two instructions of 16 rows, rows r and r + 4 of
//     8), a wavefront's loads are consecutive.  k = gate * Hp + unit, Hp = H rounded up to 4.
//   * The wavefronts' partial tiles are added through LDS in wavefront order; a thread then owns one
//     (row, unit), whose state stays in its registers.
//   * The inputs of the next step are requested behind the last operand load of a product, so that
//     they neither delay an operand nor a look at the barrier's flags.
// Bound: the chain exchange - operand load - product - pointwise math of a step (a tanh takes 0.3 us, two follow each
// other).  The matrix cores need 1.9 us of a step.
// Measured per step at N = 64, H = 512, LSTM, step-wise -> 16 rows -> 8 rows (launches of 100 steps, set-up included): forward
// 14.7 -> 6.1 -> 5.6 us, backward 14.9 -> 8.4 -> 6.4 us.  Whole training passes, 16 rows behind barriers -> now (with
// gemm_f64's changes), T = 100: LSTM N = 64, H = 512 2.70 -> 2.20 ms, GRU 2.33 -> 1.85; N = 64, H = 128 0.81 -> 0.67; GRU N = 5, H = 64 0.52 -> 0.44;
// T = 50: N = 32, H = 768 1.77 -> 1.49, N = 40, H = 700 2.52 -> 1.59.
#include "recurrent.h"

namespace haste_hip {
namespace {

typedef unsigned int uint2_t __attribute__((ext_vector_type(2)));
typedef double double2_t __attribute__((ext_vector_type(2)));
typedef double double4_t __attribute__((ext_vector_type(4)));
constexpr unsigned int kNowhere64 = 0x7ffffff0u;  // beyond any buffer resource's range: the load returns zeros
constexpr int kChunk64 = 8;  // instructions whose operands are requested together
constexpr int kAgentScope64 = 16;  // the sc1 bit of a load's cache policy

constexpr __host__ __device__ int rounded_up(int x, int m) { return (x + m - 1) / m * m; }

__device__ __forceinline__ double sigmoid_d(double x) { return 1.0 / (1.0 + exp(-x)); }

__device__ __forceinline__ void store_exchanged_d(const GroupSync& g, double* p, double v) {
  if (g.same_xcd) *p = v;
  else
    __hip_atomic_store(reinterpret_cast<unsigned long long*>(p), __builtin_bit_cast(unsigned long long, v),
                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Polled tiles (recurrent.h): what has not been published holds a bit pattern that no producer stores.  An element's
// eight bytes arrive together: they are one aligned store.
__device__ __forceinline__ double unwritten_d() { return __builtin_bit_cast(double, ~0ull); }
__device__ __forceinline__ double publishable_d(double v) {
  return __builtin_bit_cast(unsigned long long, v) == ~0ull ? __builtin_bit_cast(double, 0x7ff8000000000000ull) : v;
}
__device__ __forceinline__ bool written_d(double2_t a) {
  const double x = a[0], y = a[1];  // bit_cast of an element itself takes the vector's first
  return __builtin_bit_cast(unsigned long long, x) != ~0ull && __builtin_bit_cast(unsigned long long, y) != ~0ull;
}
template <int N>
__device__ __forceinline__ bool all_written_d(const double2_t (&a)[N]) {
  bool written = true;
#pragma unroll
  for (int i = 0; i < N; ++i) written = written && written_d(a[i]);
  return __all(written) != 0;
}

// Where the A operand for contraction index k and batch row `row` of a group lies in its tile.
template <int ROWS>
__device__ __forceinline__ int exchange_index(int k, int row) {
  if (ROWS == 8) return (k * 4 + (row & 3)) * 2 + (row >> 2);
  const int s = k >> 2;
  return ((s >> 1) * 64 + (k & 3) * 16 + row) * 2 + (s & 1);
}

struct RecurrenceShape {
  LaunchShape ls;
  int T, N, H;
  int kw;                 // instructions of a wavefront per step and column tile, a multiple of kChunk64
  const double* weights;  // [kIn * H][kOut * H]
  double* exchange;       // [groups][kPolledTiles][16 * kw * rows of a group]
};

// A cell: its parameters, what a step reads of the caller's memory (Inputs, requested a step
// ahead; prepare() does what needs nothing else while the workgroup waits for the others), what a thread carries from step to step, and the arithmetic of stepwise.hip's kernels.
struct LstmForward64 {
  static constexpr bool kForward = true;
  static constexpr int kIn = 1, kOut = 4;
  struct Params : RecurrenceShape {
    int training;
    float zoneout_prob;
    const double *b, *h, *c, *mask;
    double *h_out, *c_out, *v;
  };
  struct Inputs { double a[4], m; };
  double bias[4], h, c, gate[4];

  __device__ void begin(const Params& p, size_t idx, int j) {
    h = p.h[idx];
    c = p.c[idx];
#pragma unroll
    for (int g = 0; g < 4; ++g) bias[g] = p.b[g * p.H + j];
  }
  __device__ double initial(int) const { return h; }
  __device__ void prepare(const Inputs&) {}
  __device__ static void request(const Params& p, int s, int n, int j, Inputs& in) {
    const size_t row = (size_t)s * p.N + n;
#pragma unroll
    for (int g = 0; g < 4; ++g) in.a[g] = p.v[row * 4 * p.H + (size_t)g * p.H + j];
    in.m = (p.mask != nullptr ? p.mask : p.h_out)[row * p.H + j];
  }
  __device__ void step(const Params& p, const Inputs& in, const double (&sum)[4]) {
    double a[4];
#pragma unroll
    for (int g = 0; g < 4; ++g) a[g] = in.a[g] + sum[g] + bias[g];
    gate[0] = sigmoid_d(a[0]);
    gate[1] = tanh(a[1]);
    gate[2] = sigmoid_d(a[2]);
    gate[3] = sigmoid_d(a[3]);
    c = gate[2] * c + gate[0] * gate[1];
    double h_new = gate[3] * tanh(c);
    if (p.zoneout_prob != 0.f && p.mask != nullptr) {
      if (p.training) h_new = (h_new - h) * in.m + h;
      else h_new = double(p.zoneout_prob) * h + (1.0 - double(p.zoneout_prob)) * h_new;
    }
    h = h_new;
  }
  __device__ double published(int) const { return h; }
  __device__ void store(const Params& p, int s, int n, int j) const {
    const size_t row = (size_t)s * p.N + n;
    p.h_out[row * p.H + j] = h;
    p.c_out[row * p.H + j] = c;
    if (p.training)
#pragma unroll
      for (int g = 0; g < 4; ++g) p.v[row * 4 * p.H + (size_t)g * p.H + j] = gate[g];
  }
  __device__ void finish(const Params&, size_t, const double (&)[4]) {}
};

struct GruForward64 {
  static constexpr bool kForward = true;
  static constexpr int kIn = 1, kOut = 3;
  struct Params : RecurrenceShape {
    int training;
    float zoneout_prob;
    const double *bx, *br, *h, *wx, *mask;
    double *h_out, *v;
  };
  struct Inputs { double a[3], m; };
  double bias_x[3], bias_r[3], h, gate[4];

  __device__ void begin(const Params& p, size_t idx, int j) {
    h = p.h[idx];
#pragma unroll
    for (int g = 0; g < 3; ++g) {
      bias_x[g] = p.bx[g * p.H + j];
      bias_r[g] = p.br[g * p.H + j];
    }
  }
  __device__ double initial(int) const { return h; }
  __device__ void prepare(const Inputs&) {}
  __device__ static void request(const Params& p, int s, int n, int j, Inputs& in) {
    const size_t row = (size_t)s * p.N + n;
#pragma unroll
    for (int g = 0; g < 3; ++g) in.a[g] = p.wx[row * 3 * p.H + (size_t)g * p.H + j];
    in.m = (p.mask != nullptr ? p.mask : p.h_out)[row * p.H + j];
  }
  __device__ void step(const Params& p, const Inputs& in, const double (&sum)[3]) {
    gate[0] = sigmoid_d(in.a[0] + sum[0] + bias_x[0] + bias_r[0]);
    gate[1] = sigmoid_d(in.a[1] + sum[1] + bias_x[1] + bias_r[1]);
    gate[3] = sum[2] + bias_r[2];
    gate[2] = tanh(in.a[2] + gate[1] * gate[3] + bias_x[2]);
    double h_new = gate[0] * h + (1.0 - gate[0]) * gate[2];
    if (p.zoneout_prob != 0.f && p.mask != nullptr) {
      if (p.training) h_new = (h_new - h) * in.m + h;
      else h_new = double(p.zoneout_prob) * h + (1.0 - double(p.zoneout_prob)) * h_new;
    }
    h = h_new;
  }
  __device__ double published(int) const { return h; }
  __device__ void store(const Params& p, int s, int n, int j) const {
    const size_t row = (size_t)s * p.N + n;
    p.h_out[row * p.H + j] = h;
    if (p.training)
#pragma unroll
      for (int g = 0; g < 4; ++g) p.v[row * 4 * p.H + (size_t)g * p.H + j] = gate[g];
  }
  __device__ void finish(const Params&, size_t, const double (&)[3]) {}
};

// Backward: step s is time t = T - 1 - s.  `dh` carries what bypasses the cell; the product of the
// gate gradients of the step before is added to it.
struct LstmBackward64 {
  static constexpr bool kForward = false;
  static constexpr int kIn = 4, kOut = 1;
  struct Params : RecurrenceShape {
    const double *c, *c_next, *dh_next, *dc_next, *mask;
    double *dh, *dc, *v;
  };
  struct Inputs { double gate[4], c, c_next, dh, dc, m; };
  double dh, dc, c_tanh, grad[4];

  __device__ void begin(const Params& p, size_t idx, int) {
    dh = p.dh[idx];
    dc = p.dc[idx];
  }
  __device__ double initial(int) const { return 0.0; }
  __device__ void prepare(const Inputs& in) { c_tanh = tanh(in.c_next); }
  __device__ static void request(const Params& p, int s, int n, int j, Inputs& in) {
    const size_t row = (size_t)(p.T - 1 - s) * p.N + n, at = row * p.H + j;
#pragma unroll
    for (int g = 0; g < 4; ++g) in.gate[g] = p.v[row * 4 * p.H + (size_t)g * p.H + j];
    in.c = p.c[at];
    in.c_next = p.c_next[at];
    in.dh = p.dh_next[at];
    in.dc = (p.dc_next != nullptr ? p.dc_next : p.dh_next)[at];
    in.m = (p.mask != nullptr ? p.mask : p.dh_next)[at];
  }
  __device__ void step(const Params& p, const Inputs& in, const double (&sum)[1]) {
    double dc_total = (p.dc_next != nullptr ? in.dc : 0.0) + dc;
    double dh_total = in.dh + (dh + sum[0]);
    dh = 0.0;
    if (p.mask != nullptr) {
      dh = (1.0 - in.m) * dh_total;
      dh_total = in.m * dh_total;
    }
    const double gi = in.gate[0], gg = in.gate[1], gf = in.gate[2], go = in.gate[3];
    const double d_o = c_tanh * dh_total;
    dc_total += (1.0 - c_tanh * c_tanh) * (go * dh_total);
    const double d_f = in.c * dc_total, d_i = gg * dc_total, d_g = gi * dc_total;
    dc = gf * dc_total;
    grad[0] = gi * (1.0 - gi) * d_i;
    grad[1] = (1.0 - gg * gg) * d_g;
    grad[2] = gf * (1.0 - gf) * d_f;
    grad[3] = go * (1.0 - go) * d_o;
  }
  __device__ double published(int g) const { return grad[g]; }
  __device__ void store(const Params& p, int s, int n, int j) const {
    const size_t row = (size_t)(p.T - 1 - s) * p.N + n;
#pragma unroll
    for (int g = 0; g < 4; ++g) p.v[row * 4 * p.H + (size_t)g * p.H + j] = grad[g];
  }
  __device__ void finish(const Params& p, size_t idx, const double (&sum)[1]) {
    p.dh[idx] = dh + sum[0];
    p.dc[idx] = dc;
  }
};

struct GruBackward64 {
  static constexpr bool kForward = false;
  static constexpr int kIn = 3, kOut = 1;
  struct Params : RecurrenceShape {
    const double *h, *v, *dh_next, *mask;
    double *dh, *dp, *dq;
  };
  struct Inputs { double gate[4], h, dh, m; };
  double dh, grad[3], dp_g;

  __device__ void begin(const Params& p, size_t idx, int) { dh = p.dh[idx]; }
  __device__ double initial(int) const { return 0.0; }
  __device__ void prepare(const Inputs&) {}
  __device__ static void request(const Params& p, int s, int n, int j, Inputs& in) {
    const size_t row = (size_t)(p.T - 1 - s) * p.N + n, at = row * p.H + j;
#pragma unroll
    for (int g = 0; g < 4; ++g) in.gate[g] = p.v[row * 4 * p.H + (size_t)g * p.H + j];
    in.h = p.h[at];
    in.dh = p.dh_next[at];
    in.m = (p.mask != nullptr ? p.mask : p.dh_next)[at];
  }
  __device__ void step(const Params& p, const Inputs& in, const double (&sum)[1]) {
    const double z = in.gate[0], r = in.gate[1], g = in.gate[2], qg = in.gate[3];
    double dh_total = in.dh + (dh + sum[0]);
    if (p.mask != nullptr) {
      dh = (1.0 - in.m) * dh_total;
      dh_total = in.m * dh_total;
      dh += z * dh_total;
    } else {
      dh = z * dh_total;
    }
    const double dg = (1.0 - z) * dh_total, dz = (in.h - g) * dh_total;
    dp_g = (1.0 - g * g) * dg;
    grad[2] = dp_g * r;
    grad[1] = r * (1.0 - r) * (dp_g * qg);
    grad[0] = z * (1.0 - z) * dz;
  }
  __device__ double published(int g) const { return grad[g]; }
  __device__ void store(const Params& p, int s, int n, int j) const {
    const size_t at = ((size_t)(p.T - 1 - s) * p.N + n) * 3 * p.H + j;
    p.dp[at] = p.dq[at] = grad[0];
    p.dp[at + p.H] = p.dq[at + p.H] = grad[1];
    p.dp[at + 2 * (size_t)p.H] = dp_g;
    p.dq[at + 2 * (size_t)p.H] = grad[2];
  }
  __device__ void finish(const Params& p, size_t idx, const double (&sum)[1]) { p.dh[idx] = dh + sum[0]; }
};

// The kernels' KS: the smallest that holds kw serves it.
constexpr int kSteps64[] = {8, 16, 32, 48, 64, 96, 128, 160, 192};
constexpr int smaller_steps64(int ks) {
  int before = 0;
  for (int s : kSteps64)
    if (s < ks) before = s;
  return before;
}
constexpr int column_tiles64(int gates, int units) { return (gates * units + 15) / 16; }

// Of a wavefront's ks instructions per column tile, those whose weights lie in LDS: what leaves at
// most 64 doubles per lane in registers (with all 128 of a backward step at H = 512 there, four chunks
// of operands in flight are spilled: 12.7 us per step, two chunks 9.5, this 8.4), as far as LDS reaches beside the partial tiles.
constexpr int lds_steps64(int ks, int ct, int rows) {
  int steps = 0;
  while ((ks - steps) * ct > 64 && (steps + kChunk64) * ct * 2048 + ct * rows * 512 + 16 <= (int)kMaxLdsBytes) steps += kChunk64;
  return steps;
}
constexpr bool fits64(int ks, int ct, int rows) { return (ks - lds_steps64(ks, ct, rows)) * ct <= 128; }
// Partial tiles of the four wavefronts, one word for the role, the weights in LDS.
constexpr size_t recurrence64_lds_bytes(int ks, int ct, int rows) {
  return (size_t)ct * rows * 512 + 16 + (size_t)lds_steps64(ks, ct, rows) * ct * 2048;
}

// Lanes of a row of 16: the value of the lane 4 * BLOCKS before (in a circle), BLOCKS = 1 only for lanes whose bit 2 is
// set, the others the lane 4 behind: the neighbour block.
template <int CTRL, int BANKS>
__device__ __forceinline__ unsigned int moved(unsigned int old, unsigned int v) {
  return (unsigned int)__builtin_amdgcn_update_dpp((int)old, (int)v, CTRL, 0xf, BANKS, false);
}
__device__ __forceinline__ double from_block(double v, bool two) {
  const uint2_t x = __builtin_bit_cast(uint2_t, v);
  uint2_t y;
#pragma unroll
  for (int i = 0; i < 2; ++i)
    y[i] = two ? moved<0x128, 0xf>(x[i], x[i])                               // row_ror:8
               : moved<0x12c, 0x5>(moved<0x124, 0xf>(x[i], x[i]), x[i]);     // row_ror:4, in blocks 0 and 2 row_ror:12
  return __builtin_bit_cast(double, y);
}

// Polled tiles or the step barrier.  A look at a tile costs more the longer a wavefront's share of it is, and its chunks
// arrive one after the other; the barrier costs a store's acknowledgement and a flag's round trip, more across XCDs.
// Training passes, barrier / polled, ms: 8 rows, T = 100: N = 64 H = 128 0.785 / 0.670, N = 20 H = 256 (GRU) 0.744 / 0.691,
// N = 37 H = 300 1.149 / 1.167, N = 64 H = 512 2.25 / 2.30 (inference 0.811 / 0.900); 16 rows: N = 128 H = 256
// 1.29 / 1.25, T = 50 N = 32 H = 768 1.78 / 1.49, but inference with H = 768 0.462 / 0.492.
constexpr bool polled64(bool forward, int ks, int rows) {
  return rows == 16 ? !forward || ks <= 32 : ks <= (forward ? 16 : 64);
}

template <class Cell, int HS, int KS, int ROWS>
__global__ __launch_bounds__(256, 1)
void recurrence64_kernel(typename Cell::Params p) {
  constexpr int CT = column_tiles64(Cell::kOut, HS);
  constexpr int CHAINS = CT == 1 ? 2 : 1;  // accumulators per column tile: no instruction waits for the one before
  constexpr int KL = lds_steps64(KS, CT, ROWS), KR = KS - KL;
  constexpr bool kShort = ROWS == 8;
  // Short tiles, blocks over k: "instruction" i stands for columns 4 * (i % 4) .. +3 and 16 k.
  constexpr bool kBlocksOverK = kShort && CT == 1;
  constexpr int LOADS = kBlocksOverK ? kChunk64 / 4 : kShort ? kChunk64 : kChunk64 / 2;  // 16-byte operand loads of a chunk
  // chunks of operands in registers (CT > 1: no gain)
  constexpr int RING = KS >= 4 * kChunk64 && CT == 1 ? (kShort && KS >= 8 * kChunk64 ? 8 : 4) : 2;
  constexpr bool kPolled = polled64(Cell::kForward, KS, ROWS);
  // The chunk behind whose request those of the inputs go: the last that every kw served by this KS has.
  constexpr int kInputsBehind = smaller_steps64(KS) / kChunk64;
  extern __shared__ double partial[];
  const Role role = take_role(p.ls, reinterpret_cast<unsigned int*>(partial + CT * ROWS * 64));
  if (!role.active) return;
  GroupSync gs;
  group_sync_init(gs, p.ls, role);
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 15, q = lane >> 4;
  const int H = p.H, Hp = rounded_up(H, 4), kw = p.kw;

  double w[KR][CT];
  double2_t* w_lds = reinterpret_cast<double2_t*>(partial + CT * ROWS * 64 + 2) + (size_t)wave * (KL / 2) * CT * 64 + lane;
  {
    const int row_len = Cell::kOut * H;
    const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<double*>(p.weights), 0, Cell::kIn * H * row_len * 8, 0x00020000);
#pragma unroll
    for (int i = 0; i < KS; ++i) {
      const int k = kBlocksOverK ? 4 * wave * kw + 16 * (i / 4) + (lane >> 2) : 4 * (wave * kw + i) + q;
      const int gate = k / Hp, unit = k % Hp;
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) {
        const int col = kBlocksOverK ? 4 * (i % 4) + (lane & 3) : 16 * ct + c, out = col / HS, owned = role.cw * HS + col % HS;
        const bool there = i < kw && gate < Cell::kIn && unit < H && out < Cell::kOut && owned < H;
        const unsigned int off = there ? (unsigned int)(((gate * H + unit) * row_len + out * H + owned) * 8) : kNowhere64;
        const double v = __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(rw, off, 0, 0));
        if (i < KR) w[i < KR ? i : 0][ct] = v;
        else w_lds[((i - KR) / 2 * CT + ct) * 64][i % 2] = v;  // read by this lane only
      }
    }
  }

  const int tile = 16 * kw * ROWS;
  double* exchange = p.exchange + (size_t)role.bt * kPolledTiles * tile;
  for (int i = role.cw * 256 + tid; i < kPolledTiles * tile; i += p.ls.gx * 256) store_exchanged_d(gs, exchange + i, 0.0);
  group_arrive(gs);
  group_wait(gs);

  const int u = tid % HS, row = tid / HS;
  const int n = role.bt * ROWS + row, j = role.cw * HS + u;
  const bool owner = row < ROWS && n < p.N && j < H;
  const size_t idx = (size_t)n * H + j;
  // Requests are unconditional (a branch would make every wait behind it a wait for all loads: 9.5
  // instead of 8.4 us per backward step): threads without an element read the last one's.
  const int n_read = n < p.N ? n : p.N - 1, j_read = j < H ? j : H - 1;
  const int last_step = p.T - 1;  // the backward loop's turn T, which only adds the last product, has no inputs
  Cell cell;
  typename Cell::Inputs in, next;
  Cell::request(p, 0, n_read, j_read, in);
  if (owner) {
    cell.begin(p, idx, j);
    // Tile 0 receives the initial state; the others' elements that steps will publish start out unwritten.
    for (int g = 0; g < Cell::kIn; ++g)
      for (int b = 0; b < kPolledTiles; ++b)
        store_exchanged_d(gs, exchange + b * tile + exchange_index<ROWS>(g * Hp + j, row),
                          Cell::kForward && b == 0 ? publishable_d(cell.initial(0)) : unwritten_d());
  }
  group_arrive(gs);
  if constexpr (kPolled) group_wait(gs);

  for (int s = 0; s <= p.T; ++s) {
    if (Cell::kForward && s == p.T) break;
    double sum[Cell::kOut] = {};
    if (owner) cell.prepare(in);
    if (Cell::kForward || s > 0) {
      const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc(
          exchange + (size_t)(s % kPolledTiles) * tile, 0, tile * 8, 0x00020000);
      // Short tiles: rows r and r + 4 of a k side by side, 256 bytes per 4 k; with blocks over columns every block
      // reads the same.
      const unsigned int base = kBlocksOverK ? (unsigned int)(wave * kw * 256 + lane * 16)
                                : kShort     ? (unsigned int)(wave * kw * 256 + (q * 4 + (lane & 3)) * 16)
                                             : (unsigned int)(wave * kw / 2 * 64 + lane) * 16u;
      constexpr int kStride = kShort && !kBlocksOverK ? 256 : 1024;
      double2_t a[RING][LOADS];
      auto request_one = [&](int set, int first, int i) {
        a[set][i] = __builtin_bit_cast(double2_t, __builtin_amdgcn_raw_buffer_load_b128(
                                                      ra, base, (first / kChunk64 * LOADS + i) * kStride, kAgentScope64));
      };
      auto request = [&](int set, int first) {
        if (first >= kw) first = 0;  // nobody uses it; a load that is always there keeps the waits exact
#pragma unroll
        for (int i = 0; i < LOADS; ++i) request_one(set, first, i);
      };
      // Waits for a chunk: what is missing is asked for again.  The loop is apart from the first look, so that this one
      // waits for its chunk only.
      auto arrive = [&](int set, int first) {
        if (kPolled && !all_written_d(a[set]))
          poll_until_written(gs, [&] {
#pragma unroll
            for (int i = 0; i < LOADS; ++i)
              if (__all(written_d(a[set][i])) == 0) request_one(set, first, i);
          }, [&] { return all_written_d(a[set]); });
      };
      if constexpr (!kPolled) group_wait(gs);
      request(0, 0);
      arrive(0, 0);  // the first chunk tells when the others are worth asking for: most of what is to come arrives at one time
#pragma unroll
      for (int ch = 1; ch < RING - 1; ++ch) request(ch, ch * kChunk64);
      auto chunks = [&](auto&& multiply) {
#pragma unroll
        for (int ch = 0; ch < KS / kChunk64; ++ch) {
          if (ch * kChunk64 >= kw) break;
          if (ch > 0) arrive(ch % RING, ch * kChunk64);
          if (ch + RING - 1 < KS / kChunk64) request((ch + RING - 1) % RING, (ch + RING - 1) * kChunk64);
          if (ch == kInputsBehind) Cell::request(p, s < last_step ? s + 1 : last_step, n_read, j_read, next);
#pragma unroll
          for (int i = 0; i < kChunk64; i += 2)
#pragma unroll
            for (int ct = 0; ct < CT; ++ct) {
              const int k = ch * kChunk64 + i;
              const double2_t b = k < KR ? double2_t{w[k < KR ? k : 0][ct], w[k < KR ? k + 1 : 0][ct]}
                                         : w_lds[((k - KR) / 2 * CT + ct) * 64];
              multiply(a[ch % RING], i, ct, b);
            }
        }
      };
      if constexpr (kShort) {
        constexpr int OUTS = kBlocksOverK ? 4 : CT;
        double acc[OUTS][2];
#pragma unroll
        for (int g = 0; g < OUTS; ++g) acc[g][0] = acc[g][1] = 0.0;
        chunks([&](const double2_t (&x)[LOADS], int i, int ct, double2_t b) {
#pragma unroll
          for (int e = 0; e < 2; ++e) {
            const int g = kBlocksOverK ? (i + e) % 4 : ct, load = kBlocksOverK ? (i + e) / 4 : i + e;
#pragma unroll
            for (int r = 0; r < 2; ++r) acc[g][r] = __builtin_amdgcn_mfma_f64_4x4x4f64(x[load][r], b[e], acc[g][r], 0, 0, 0);
          }
        });
        if constexpr (kBlocksOverK) {
          // The four blocks' sums are added where the columns belong: block b keeps columns 4 b .. 4 b + 3.
          const bool upper = (lane & 8) != 0, odd = (lane & 4) != 0;
#pragma unroll
          for (int r = 0; r < 2; ++r) {
            const double a0 = (upper ? acc[2][r] : acc[0][r]) + from_block(upper ? acc[0][r] : acc[2][r], true);
            const double a1 = (upper ? acc[3][r] : acc[1][r]) + from_block(upper ? acc[1][r] : acc[3][r], true);
            partial[wave * ROWS * 16 + (4 * r + q) * 16 + c] = (odd ? a1 : a0) + from_block(odd ? a0 : a1, false);
          }
        } else {
#pragma unroll
          for (int ct = 0; ct < CT; ++ct)
#pragma unroll
            for (int r = 0; r < 2; ++r) partial[(wave * CT + ct) * ROWS * 16 + (4 * r + q) * 16 + c] = acc[ct][r];
        }
      } else {
        double4_t acc[CT][CHAINS];
#pragma unroll
        for (int ct = 0; ct < CT; ++ct)
#pragma unroll
          for (int e = 0; e < CHAINS; ++e) acc[ct][e] = double4_t{0.0, 0.0, 0.0, 0.0};
        chunks([&](const double2_t (&x)[LOADS], int i, int ct, double2_t b) {
          acc[ct][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(x[i / 2][0], b[0], acc[ct][0], 0, 0, 0);
          acc[ct][CHAINS - 1] = __builtin_amdgcn_mfma_f64_16x16x4f64(x[i / 2][1], b[1], acc[ct][CHAINS - 1], 0, 0, 0);
        });
#pragma unroll
        for (int ct = 0; ct < CT; ++ct)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            double v = acc[ct][0][r];
            if (CHAINS == 2) v += acc[ct][CHAINS - 1][r];
            partial[(wave * CT + ct) * 256 + (4 * r + q) * 16 + c] = v;
          }
      }
      __syncthreads();
      if (row < ROWS) {
#pragma unroll
        for (int g = 0; g < Cell::kOut; ++g) {
          constexpr int TILE = ROWS * 16, WAVE = CT * TILE;
          const int col = g * HS + u, at = (col / 16) * TILE + row * 16 + col % 16;
          sum[g] = ((partial[at] + partial[WAVE + at]) + partial[2 * WAVE + at]) + partial[3 * WAVE + at];
        }
      }
    } else {
      Cell::request(p, s < last_step ? s + 1 : last_step, n_read, j_read, next);
    }
    if (!Cell::kForward && s == p.T) {
      if (owner) cell.finish(p, idx, sum);
      break;
    }
    if (owner) cell.step(p, in, sum);
    // What this wavefront stored during the step before (its resets among it) has landed before the step is visible.
    if constexpr (kPolled) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if (owner && (!Cell::kForward || s + 1 < p.T)) {
      double* to = exchange + (size_t)((s + 1) % kPolledTiles) * tile;
      double* done = exchange + (size_t)((s + 3) % kPolledTiles) * tile;  // read at step s - 1: nobody needs it any more
#pragma unroll
      for (int g = 0; g < Cell::kIn; ++g) {
        const int e = exchange_index<ROWS>(g * Hp + j, row);
        store_exchanged_d(gs, to + e, kPolled ? publishable_d(cell.published(g)) : cell.published(g));
        if constexpr (kPolled) store_exchanged_d(gs, done + e, unwritten_d());
      }
    }
    if constexpr (kPolled) __syncthreads();  // the partial tiles may be overwritten
    else group_arrive(gs);
    if (owner) cell.store(p, s, n, j);
    in = next;
  }
}

// The geometry: rows of a group, HS units per workgroup, what a wavefront does per step.
struct Plan64 { int rows, hs, gx, gy, kw; };

// The kernels there are: those whose weights fit registers and LDS, groups of 8 rows as far as the plan below has a use
// for them.
constexpr bool offered64(bool forward, int hs, int ks, int rows, int ct) {
  return fits64(ks, ct, rows) && (rows == 16 || ks <= (forward ? (hs == 16 ? 48 : 16) : 128));
}
// The kernel's KS for kw instructions per wavefront and column tile, 0 when there is none.
constexpr int variant64(bool forward, int hs, int kw, int rows, int ct) {
  for (int ks : kSteps64)
    if (kw <= ks) return offered64(forward, hs, ks, rows, ct) ? ks : 0;
  return 0;
}

// Groups of 8 rows where each has an XCD of its own, otherwise of 16 rows, which need half the
// workgroups, or 8 across XCDs where those are the only ones whose weights fit; 16 hidden units per workgroup unless 8
// are offered and fit.  The weights of a wavefront must fit its registers and its part of LDS.
bool plan_recurrence64(int in_gates, int out_gates, int N, int H, bool eight_units, Plan64* plan) {
  const int steps = in_gates * rounded_up(H, 4) / 4;
  plan->kw = rounded_up((steps + 3) / 4, kChunk64);
  for (int choice = 0; choice < 3; ++choice)
    for (int hs : {8, 16}) {
      if (hs == 8 && (!eight_units || choice == 2)) continue;
      plan->rows = choice == 1 ? 16 : 8;
      plan->hs = hs;
      plan->gx = (H + hs - 1) / hs;
      plan->gy = (N + plan->rows - 1) / plan->rows;
      if (choice == 0 && !xcd_local_fits(plan->gx, plan->gy)) continue;
      if (choice == 2 && in_gates > 1) continue;
      if (variant64(out_gates > 1, hs, plan->kw, plan->rows, column_tiles64(out_gates, hs)) > 0 && plan->gy <= kMaxGroups &&
          (long long)plan->gx * plan->gy <= device_cu_count() && plan->gx * plan->gy <= kMaxWorkgroups)
        return true;
    }
  return false;
}

// Room for groups of 8 rows and of 16: which of them run is asked again at the launch, and another thread may have found
// the placement on XCDs wrong in between.
size_t exchange64_bytes(const Plan64& plan, int N) {
  return (size_t)rounded_up(N, 16) * kPolledTiles * 16 * plan.kw * sizeof(double);
}

template <class Cell, int HS, int ROWS>
int launch_recurrence64(const char* name, hipStream_t stream, const Plan64& plan, typename Cell::Params& p) {
  constexpr int CT = column_tiles64(Cell::kOut, HS);
  Workspace ws;
  HASTE_HIP_PROPAGATE(get_workspace(stream, 0, &ws));
  HASTE_HIP_PROPAGATE(check_and_clear_abort(stream, &ws));
  LaunchPlan launch;
  const int variant = variant64(Cell::kForward, HS, plan.kw, ROWS, CT);
  HASTE_HIP_PROPAGATE(plan_launch(stream, ws, plan.gx, plan.gy, ROWS, recurrence64_lds_bytes(variant, CT, ROWS),
                                  (unsigned)p.T + 3, &launch));
  p.ls = launch.shape;
  launch.kernel = kPlanDouble;
  p.kw = plan.kw;
#define HASTE_LAUNCH_64(KS_)                                   \
  if constexpr (offered64(Cell::kForward, HS, KS_, ROWS, CT))  \
    if (variant == KS_) return launch_persistent(name, recurrence64_kernel<Cell, HS, KS_, ROWS>, launch, p, stream);
  HASTE_LAUNCH_64(8) HASTE_LAUNCH_64(16) HASTE_LAUNCH_64(32) HASTE_LAUNCH_64(48) HASTE_LAUNCH_64(64)
  HASTE_LAUNCH_64(96) HASTE_LAUNCH_64(128) HASTE_LAUNCH_64(160) HASTE_LAUNCH_64(192)
#undef HASTE_LAUNCH_64
  return HASTE_HIP_ERROR_UNSUPPORTED_SIZE;
}

template <class Cell>
int launch_recurrence64(const char* name, hipStream_t stream, const Plan64& plan, typename Cell::Params& p) {
  if constexpr (Cell::kForward)
    if (plan.hs == 8) return plan.rows == 8 ? launch_recurrence64<Cell, 8, 8>(name, stream, plan, p)
                                            : launch_recurrence64<Cell, 8, 16>(name, stream, plan, p);
  return plan.rows == 8 ? launch_recurrence64<Cell, 16, 8>(name, stream, plan, p)
                        : launch_recurrence64<Cell, 16, 16>(name, stream, plan, p);
}

}  // namespace

// Bytes of scratch the recurrence needs in one launch, 0 when it runs step by step.  A launch
// costs its set-up (the weights, two barriers: about 10 us), as much as a step of its own: from
// four steps on.  `in_gates` / `out_gates`: blocks of H in the contraction and in its result.
size_t recurrence64_scratch_bytes(int in_gates, int out_gates, int steps, int N, int H) {
  Plan64 plan;
  if (steps < 4 || !plan_recurrence64(in_gates, out_gates, N, H, out_gates > 1, &plan)) return 0;
  return exchange64_bytes(plan, N);
}

int lstm_forward_recurrence64(hipStream_t stream, int training, int T, int N, int H, const double* R, const double* b,
                              const double* h, const double* c, double* h_out, double* c_out, double* v,
                              float zoneout_prob, const double* mask, void* exchange) {
  Plan64 plan;
  if (!plan_recurrence64(1, 4, N, H, true, &plan)) return HASTE_HIP_ERROR_UNSUPPORTED_SIZE;
  LstmForward64::Params p = {};
  p.T = T; p.N = N; p.H = H; p.weights = R; p.exchange = static_cast<double*>(exchange);
  p.training = training; p.zoneout_prob = zoneout_prob; p.mask = mask;
  p.b = b; p.h = h; p.c = c; p.h_out = h_out; p.c_out = c_out; p.v = v;
  const char* name = "lstm_forward_recurrence64";
  return launch_recurrence64<LstmForward64>(name, stream, plan, p);
}

int gru_forward_recurrence64(hipStream_t stream, int training, int T, int N, int H, const double* R, const double* bx,
                             const double* br, const double* h, const double* wx, double* h_out, double* v,
                             float zoneout_prob, const double* mask, void* exchange) {
  Plan64 plan;
  if (!plan_recurrence64(1, 3, N, H, true, &plan)) return HASTE_HIP_ERROR_UNSUPPORTED_SIZE;
  GruForward64::Params p = {};
  p.T = T; p.N = N; p.H = H; p.weights = R; p.exchange = static_cast<double*>(exchange);
  p.training = training; p.zoneout_prob = zoneout_prob; p.mask = mask;
  p.bx = bx; p.br = br; p.h = h; p.wx = wx; p.h_out = h_out; p.v = v;
  const char* name = "gru_forward_recurrence64";
  return launch_recurrence64<GruForward64>(name, stream, plan, p);
}

int lstm_backward_recurrence64(hipStream_t stream, int T, int N, int H, const double* R_t, const double* c,
                               const double* c_next, const double* dh_next, const double* dc_next, double* dh,
                               double* dc, double* v, const double* mask, void* exchange) {
  Plan64 plan;
  if (!plan_recurrence64(4, 1, N, H, false, &plan)) return HASTE_HIP_ERROR_UNSUPPORTED_SIZE;
  LstmBackward64::Params p = {};
  p.T = T; p.N = N; p.H = H; p.weights = R_t; p.exchange = static_cast<double*>(exchange);
  p.c = c; p.c_next = c_next; p.dh_next = dh_next; p.dc_next = dc_next; p.mask = mask;
  p.dh = dh; p.dc = dc; p.v = v;
  return launch_recurrence64<LstmBackward64>("lstm_backward_recurrence64", stream, plan, p);
}

int gru_backward_recurrence64(hipStream_t stream, int T, int N, int H, const double* R_t, const double* h,
                              const double* v, const double* dh_next, double* dh, double* dp, double* dq,
                              const double* mask, void* exchange) {
  Plan64 plan;
  if (!plan_recurrence64(3, 1, N, H, false, &plan)) return HASTE_HIP_ERROR_UNSUPPORTED_SIZE;
  GruBackward64::Params p = {};
  p.T = T; p.N = N; p.H = H; p.weights = R_t; p.exchange = static_cast<double*>(exchange);
  p.h = h; p.v = v; p.dh_next = dh_next; p.mask = mask;
  p.dh = dh; p.dp = dp; p.dq = dq;
  return launch_recurrence64<GruBackward64>("gru_backward_recurrence64", stream, plan, p);
}

}  // namespace haste_hip
