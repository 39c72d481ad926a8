// What the LSTM's recurrence kernels are given, and the pointwise steps for those that are written for any cell.
#pragma once

#include "recurrent.h"

namespace haste_hip {
namespace {

struct LstmFwdParams {
  int training, T, N, H;
  const float* R;       // [H,4H]
  const float* b;       // [4H]
  const float* h;       // [N,H] state before the first step
  const float* c;       // [N,H]
  float* h_out;         // [T,N,H] states after each step (may start at h + N*H)
  float* c_out;         // [T,N,H]
  float* v;             // [T,N,4H] in: x*W, out (training): activations
  float zoneout_prob;
  const float* zoneout_mask;   // [T,N,H] or null
  const float* dc_mask;        // DropConnect mask [H,4H] or null
  float dc_scale;
  float* xh;                   // polled exchange tiles of h: [batch tiles][4][Kpad/4][NB][4]
  // kernels that compute the input projection themselves (XSG > 0): v does not hold x*W
  const float* x;              // [T,N,C]
  const float* W;              // [C,4H]
  int C;
  LaunchShape ls;
};

struct LstmBwdParams {
  int T, N, H;
  const float* R_t;     // [4H,H]
  const float* c;       // [T,N,H] cell state before each step
  const float* c_next;  // [T,N,H] cell state after each step (may be c + N*H)
  const float* dh_next; // [T,N,H] upstream gradient of the h each step produced
  const float* dc_next; // [T,N,H] same for c; without dc_given some tensor of that shape, not used
  int dc_given;
  float* db;            // [4H] accumulated
  float* dh;            // [N,H] in/out
  float* dc;            // [N,H] in/out
  float* v;             // [T,N,4H] in: activations, out: gate gradients
  const float* zoneout_mask;
  float* db_partial;    // [batch tiles, 4H] scratch
  float* xdv;           // polled exchange tiles of the gate gradients: [batch tiles][4][Kpad/4][NB][4]
                        // (scattered form: the pieces of partial sums, see the kernel)
  LaunchShape ls;
};

// The LSTM's pointwise forward step for the recurrence on the bf16 matrix cores (split_forward.h):
// arithmetic as in lstm_forward_kernel.
struct LstmForwardCell {
  using Params = LstmFwdParams;
  static constexpr int kGates = 4;
  static constexpr int kOut = 6, kStates = 2;  // h, c, activations (4 gates)
  float h, c, bias[4], gate[4];

  __device__ __forceinline__ void load_state(const Params& p, size_t row, size_t unit, bool mine) {
    const size_t e = row * p.H + unit;
    h = mine ? p.h[e] : 0.f;
    c = mine ? p.c[e] : 0.f;
#pragma unroll
    for (int g = 0; g < 4; ++g) bias[g] = p.b[(size_t)g * p.H + unit];
  }
  __host__ __device__ __forceinline__ static bool aligned(const Params& p) {
    return ((reinterpret_cast<uintptr_t>(p.v) | reinterpret_cast<uintptr_t>(p.h_out) | reinterpret_cast<uintptr_t>(p.c_out) |
             reinterpret_cast<uintptr_t>(p.zoneout_mask)) & 15u) == 0;
  }
  __device__ __forceinline__ static const float* in_row(const Params& p, int gate, size_t row) {
    return p.v + (row * 4 + gate) * p.H;
  }
  __device__ __forceinline__ static size_t in_stride(const Params& p) { return (size_t)p.N * 4 * p.H; }
  __device__ __forceinline__ static float* out_row(const Params& p, int i, size_t row) {
    return i == 0 ? p.h_out + row * p.H : (i == 1 ? p.c_out + row * p.H : p.v + (row * 4 + i - 2) * p.H);
  }
  __device__ __forceinline__ static size_t out_stride(const Params& p, int i) { return (size_t)p.N * p.H * (i < 2 ? 1 : 4); }
  __device__ __forceinline__ float out(int i) const { return i == 0 ? h : (i == 1 ? c : gate[i - 2]); }
  static constexpr int kCarried = 2;  // from step to step; the first one is what the product reads
  __device__ __forceinline__ float& carried(int i) { return i == 0 ? h : c; }
  __device__ __forceinline__ void step(const Params& p, const float4_t& in, float mask, const float4_t& rh, bool zoneout) {
    float a[4];
#pragma unroll
    for (int g = 0; g < 4; ++g) a[g] = in[g] + rh[g] + bias[g];
    gates_f<4, 0b0010>(a, gate);
    c = gate[2] * c + gate[0] * gate[1];
    float h_new = gate[3] * tanh_f(c);
    if (zoneout) {
      if (p.training) h_new = (h_new - h) * mask + h;
      else h_new = p.zoneout_prob * h + (1.0f - p.zoneout_prob) * h_new;
    }
    h = h_new;
  }
};

// The LSTM's pointwise backward step for the scattered form of the recurrence
// (scatter_backward.h): arithmetic as in lstm_backward_kernel.
struct LstmScatterCell {
  using Params = LstmBwdParams;
  static constexpr int kGates = 4;
  static constexpr int kInputs = 9;  // v (4 gates), c before and after, dh_next, dc_next, mask
  static constexpr int kSums = 4;
  float dh, dc, dh_keep;
  bool dc_given;
  float gi, gg, gf, go, c0, dhn, m, c_tanh, k_c, k_i, k_g, k_f, k_o, dc_total;

  __device__ __forceinline__ static float* pieces(const Params& p) { return p.xdv; }
  __device__ __forceinline__ static void request(const Params& p, float (&in)[kInputs], size_t e, size_t ve,
                                                 bool zoneout) {
    const float* vt = p.v + ve;
#pragma unroll
    for (int g = 0; g < 4; ++g) in[g] = vt[g * (size_t)p.H];
    in[4] = p.c[e];
    in[5] = p.c_next[e];
    in[6] = p.dh_next[e];
    in[7] = p.dc_next[e];
    if (zoneout) in[8] = p.zoneout_mask[e];
  }
  __device__ __forceinline__ void load_state(const Params& p, size_t e, bool mine) {
    dh = mine ? p.dh[e] : 0.f;
    dc = mine ? p.dc[e] : 0.f;
    dc_given = p.dc_given != 0;
    dh_keep = 0.f;
  }
  __device__ __forceinline__ void store_state(const Params& p, size_t e) const {
    p.dh[e] = dh;
    p.dc[e] = dc;
  }
  __device__ __forceinline__ void prepare(const float (&sv)[kInputs]) {
    gi = sv[0]; gg = sv[1]; gf = sv[2]; go = sv[3];
    c0 = sv[4]; dhn = sv[6]; m = sv[8];
    c_tanh = tanh_f(sv[5]);
    k_c = d_tanh_f(c_tanh);
    k_i = d_sigmoid_f(gi);
    k_g = d_tanh_f(gg);
    k_f = d_sigmoid_f(gf);
    k_o = d_sigmoid_f(go);
    dc_total = (dc_given ? sv[7] : 0.f) + dc;
  }
  __device__ __forceinline__ void add_gathered(float sum) { dh = dh_keep + sum; }
  __device__ __forceinline__ float4_t step(bool act, bool zoneout, float (&sums)[kSums]) {
    float4_t dv = {0.f, 0.f, 0.f, 0.f};
    dh_keep = 0.f;
    if (act) {
      float dh_total = dhn + dh;
      if (zoneout) {
        dh_keep = (1.0f - m) * dh_total;
        dh_total = m * dh_total;
      }
      const float do_ = c_tanh * dh_total;
      const float dc_tanh = go * dh_total;
      dc_total += k_c * dc_tanh;
      const float df = c0 * dc_total;
      dc = gf * dc_total;
      const float di = gg * dc_total;
      const float dg = gi * dc_total;
      dv = float4_t{k_i * di, k_g * dg, k_f * df, k_o * do_};
#pragma unroll
      for (int g = 0; g < 4; ++g) sums[g] += dv[g];
    }
    return dv;
  }
  __device__ __forceinline__ static void store_copy(const Params& p, int t, size_t n, size_t j, const float4_t& a) {
    float* vt = p.v + ((size_t)t * p.N + n) * 4 * p.H + j;
#pragma unroll
    for (int g = 0; g < 4; ++g) vt[g * (size_t)p.H] = a[g];
  }
  __device__ __forceinline__ static void add_sums(const Params& p, int col, float s) { p.db[col] += s; }

  // For split_backward_kernel.
  static constexpr int kOut = 4;
  __device__ __forceinline__ static int out_value(int i) { return i; }
  __host__ __device__ __forceinline__ static bool aligned(const Params& p) {
    return ((reinterpret_cast<uintptr_t>(p.v) | reinterpret_cast<uintptr_t>(p.c) | reinterpret_cast<uintptr_t>(p.c_next) |
             reinterpret_cast<uintptr_t>(p.dh_next) | reinterpret_cast<uintptr_t>(p.dc_next) |
             reinterpret_cast<uintptr_t>(p.zoneout_mask)) & 15u) == 0;
  }
  __device__ __forceinline__ static bool in_used(const Params& p, int i, bool zoneout) {
    return i < 7 || (i == 7 ? p.dc_given != 0 : zoneout);
  }
  __device__ __forceinline__ static const float* in_row(const Params& p, int i, size_t row) {
    if (i < 4) return p.v + (row * 4 + i) * p.H;
    return (i == 4 ? p.c : (i == 5 ? p.c_next : (i == 6 ? p.dh_next : (i == 7 ? p.dc_next : p.zoneout_mask)))) + row * p.H;
  }
  __device__ __forceinline__ static size_t in_stride(const Params& p, int i) { return (size_t)p.N * p.H * (i < 4 ? 4 : 1); }
  __device__ __forceinline__ static float* out_row(const Params& p, int i, size_t row) { return p.v + (row * 4 + i) * p.H; }
  __device__ __forceinline__ static size_t out_stride(const Params& p, int) { return (size_t)p.N * p.H * 4; }

  // For cut_recurrence_kernel: what is carried from step to step (the cell state after a step is the one before the step
  // that follows it), and the inputs that are read.
  static constexpr int kCarried = 3;
  float c_after;
  __device__ __forceinline__ float& carried(int i) { return i == 0 ? dh_keep : (i == 1 ? dc : c_after); }
  __device__ __forceinline__ void load_carried(const Params& p, size_t e, bool mine) {
    load_state(p, e, mine);
    dh_keep = dh;
    c_after = mine ? p.c_next[(size_t)(p.T - 1) * p.N * p.H + e] : 0.f;
  }
  static constexpr int kCutInputs = kInputs - 1;
  __device__ __forceinline__ static int cut_input(int i) { return i < 5 ? i : i + 1; }
  __device__ __forceinline__ void carry_inputs(float (&sv)[kInputs]) {
    sv[5] = c_after;
    c_after = sv[4];
  }
};

}  // namespace
}  // namespace haste_hip
