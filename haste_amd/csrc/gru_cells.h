// What the GRU's recurrence kernels are given, and the pointwise steps for those that are written for any cell.
#pragma once

#include "recurrent.h"

namespace haste_hip {
namespace {

struct GruFwdParams {
  int training, T, N, H;
  const float* R;        // [H,3H]
  const float* bx;       // [3H]
  const float* br;       // [3H]
  const float* h;        // [N,H] state before the first step
  float* h_out;          // [T,N,H] states after each step (may start at h + N*H)
  float* v;              // [T,N,4H] (training) or null
  const float* Wx;       // [T,N,3H] = x*W (kernels that compute the input projection themselves: unused)
  const float* W;        // [C,3H] and
  const float* x;        // [T,N,C], for those kernels
  int C;
  float zoneout_prob;
  const float* zoneout_mask;
  const float* dc_mask;  // DropConnect mask [H,3H] or null
  float dc_scale;
  float* xh;             // polled exchange tiles of h: [batch tiles][4][Kpad/4][NB][4]
  LaunchShape ls;
};

struct GruBwdParams {
  int T, N, H;
  const float* R_t;     // [3H,H]
  const float* h;       // [T,N,H] states before each step
  const float* v;       // [T,N,4H]
  const float* dh_next; // [T,N,H] upstream gradient of the h each step produced
  float* dbx;           // [3H] accumulated
  float* dbr;           // [3H] accumulated
  float* dh;            // [N,H] in/out
  float* dp;            // [T,N,3H]
  float* dq;            // [T,N,3H]
  const float* zoneout_mask;
  float* db_partial;    // [batch tiles, 6H] scratch
  float* xdq;           // exchange tiles of dq: [batch tiles][2][Kpad/4][NB][4]
                        // (scattered form: the pieces of partial sums, scatter_backward.h)
  LaunchShape ls;
};

// The GRU's pointwise forward step for the recurrence on the bf16 matrix cores (split_forward.h):
// arithmetic as in gru_forward_kernel.
struct GruForwardCell {
  using Params = GruFwdParams;
  static constexpr int kGates = 3;
  static constexpr int kOut = 5, kStates = 1;  // h, what the backward pass needs (4)
  float h, bxv[3], brv[3], saved[4];

  __device__ __forceinline__ void load_state(const Params& p, size_t row, size_t unit, bool mine) {
    h = mine ? p.h[row * p.H + unit] : 0.f;
#pragma unroll
    for (int g = 0; g < 3; ++g) {
      bxv[g] = p.bx[(size_t)g * p.H + unit];
      brv[g] = p.br[(size_t)g * p.H + unit];
    }
  }
  __host__ __device__ __forceinline__ static bool aligned(const Params& p) {
    return ((reinterpret_cast<uintptr_t>(p.Wx) | reinterpret_cast<uintptr_t>(p.v) | reinterpret_cast<uintptr_t>(p.h_out) |
             reinterpret_cast<uintptr_t>(p.zoneout_mask)) & 15u) == 0;
  }
  __device__ __forceinline__ static const float* in_row(const Params& p, int gate, size_t row) {
    return p.Wx + (row * 3 + gate) * p.H;
  }
  __device__ __forceinline__ static size_t in_stride(const Params& p) { return (size_t)p.N * 3 * p.H; }
  __device__ __forceinline__ static float* out_row(const Params& p, int i, size_t row) {
    return i == 0 ? p.h_out + row * p.H : p.v + (row * 4 + i - 1) * p.H;
  }
  __device__ __forceinline__ static size_t out_stride(const Params& p, int i) { return (size_t)p.N * p.H * (i < 1 ? 1 : 4); }
  __device__ __forceinline__ float out(int i) const { return i == 0 ? h : saved[i - 1]; }
  static constexpr int kCarried = 1;  // from step to step; the first one is what the product reads
  __device__ __forceinline__ float& carried(int) { return h; }
  __device__ __forceinline__ void step(const Params& p, const float4_t& in, float mask, const float4_t& rh, bool zoneout) {
    const float a[2] = {in[0] + rh[0] + bxv[0] + brv[0], in[1] + rh[1] + bxv[1] + brv[1]};
    float zr[2];
    gates_f<2, 0>(a, zr);
    const float z = zr[0], r = zr[1], qg = rh[2] + brv[2];
    const float g = tanh_f(in[2] + r * qg + bxv[2]);
    saved[0] = z;
    saved[1] = r;
    saved[2] = g;
    saved[3] = qg;
    float h_new = z * h + (1.0f - z) * g;
    if (zoneout) {
      if (p.training) h_new = (h_new - h) * mask + h;
      else h_new = p.zoneout_prob * h + (1.0f - p.zoneout_prob) * h_new;
    }
    h = h_new;
  }
};

// The GRU's pointwise backward step for the scattered form of the recurrence
// (scatter_backward.h): arithmetic as in gru_backward_kernel.  dh contracts over
// dq = (dp_z, dp_r, dq_g); the operand's fourth component carries dp_g for the caller's copy.
struct GruScatterCell {
  using Params = GruBwdParams;
  static constexpr int kGates = 3;
  static constexpr int kInputs = 7;  // v (z, r, g, q_g), h before the step, dh_next, mask
  static constexpr int kSums = 6;    // dbx (3), dbr (3)
  float dh, dh_keep;
  float z, r, g, qg, h0, dhn, m, k_g, k_r, k_z;

  __device__ __forceinline__ static float* pieces(const Params& p) { return p.xdq; }
  __device__ __forceinline__ static void request(const Params& p, float (&in)[kInputs], size_t e, size_t ve,
                                                 bool zoneout) {
    const float* vt = p.v + ve;
#pragma unroll
    for (int i = 0; i < 4; ++i) in[i] = vt[i * (size_t)p.H];
    in[4] = p.h[e];
    in[5] = p.dh_next[e];
    if (zoneout) in[6] = p.zoneout_mask[e];
  }
  __device__ __forceinline__ void load_state(const Params& p, size_t e, bool mine) {
    dh = mine ? p.dh[e] : 0.f;
    dh_keep = 0.f;
  }
  __device__ __forceinline__ void store_state(const Params& p, size_t e) const { p.dh[e] = dh; }
  __device__ __forceinline__ void prepare(const float (&sv)[kInputs]) {
    z = sv[0]; r = sv[1]; g = sv[2]; qg = sv[3];
    h0 = sv[4]; dhn = sv[5]; m = sv[6];
    k_g = d_tanh_f(g);
    k_r = d_sigmoid_f(r);
    k_z = d_sigmoid_f(z);
  }
  __device__ __forceinline__ void add_gathered(float sum) { dh = dh_keep + sum; }
  __device__ __forceinline__ float4_t step(bool act, bool zoneout, float (&sums)[kSums]) {
    float4_t a = {0.f, 0.f, 0.f, 0.f};
    dh_keep = 0.f;
    if (act) {
      float dh_total = dhn + dh;
      if (zoneout) {
        dh_keep = (1.0f - m) * dh_total;
        dh_total = m * dh_total;
        dh_keep += z * dh_total;
      } else {
        dh_keep = z * dh_total;
      }
      const float dg = (1.0f - z) * dh_total;
      const float dz = (h0 - g) * dh_total;
      const float dp_g = k_g * dg;
      const float dq_g = dp_g * r;
      const float dr = dp_g * qg;
      const float dp_r = k_r * dr;
      const float dp_z = k_z * dz;
      a = float4_t{dp_z, dp_r, dq_g, dp_g};
      sums[0] += dp_z;
      sums[1] += dp_r;
      sums[2] += dp_g;
      sums[3] += dp_z;
      sums[4] += dp_r;
      sums[5] += dq_g;
    }
    return a;
  }
  __device__ __forceinline__ static void store_copy(const Params& p, int t, size_t n, size_t j, const float4_t& a) {
    const size_t H = p.H;
    const size_t o3 = ((size_t)t * p.N + n) * 3 * H + j;
    p.dp[o3] = a[0];
    p.dp[o3 + H] = a[1];
    p.dp[o3 + 2 * H] = a[3];
    p.dq[o3] = a[0];
    p.dq[o3 + H] = a[1];
    p.dq[o3 + 2 * H] = a[2];
  }
  __device__ __forceinline__ static void add_sums(const Params& p, int col, float s) {
    if (col < 3 * p.H) p.dbx[col] += s;
    else p.dbr[col - 3 * p.H] += s;
  }

  // For split_backward_kernel.
  static constexpr int kOut = 6;  // dp, dq
  __device__ __forceinline__ static int out_value(int i) { return i < 3 ? (i == 2 ? 3 : i) : i - 3; }
  __host__ __device__ __forceinline__ static bool aligned(const Params& p) {
    return ((reinterpret_cast<uintptr_t>(p.v) | reinterpret_cast<uintptr_t>(p.h) | reinterpret_cast<uintptr_t>(p.dh_next) |
             reinterpret_cast<uintptr_t>(p.dp) | reinterpret_cast<uintptr_t>(p.dq) |
             reinterpret_cast<uintptr_t>(p.zoneout_mask)) & 15u) == 0;
  }
  __device__ __forceinline__ static bool in_used(const Params&, int i, bool zoneout) { return i < 6 || zoneout; }
  __device__ __forceinline__ static const float* in_row(const Params& p, int i, size_t row) {
    if (i < 4) return p.v + (row * 4 + i) * p.H;
    return (i == 4 ? p.h : (i == 5 ? p.dh_next : p.zoneout_mask)) + row * p.H;
  }
  __device__ __forceinline__ static size_t in_stride(const Params& p, int i) { return (size_t)p.N * p.H * (i < 4 ? 4 : 1); }
  __device__ __forceinline__ static float* out_row(const Params& p, int i, size_t row) {
    return i < 3 ? p.dp + (row * 3 + i) * p.H : p.dq + (row * 3 + i - 3) * p.H;
  }
  __device__ __forceinline__ static size_t out_stride(const Params& p, int) { return (size_t)p.N * p.H * 3; }

  // For cut_recurrence_kernel (see LstmScatterCell).
  static constexpr int kCarried = 1;
  __device__ __forceinline__ float& carried(int) { return dh_keep; }
  __device__ __forceinline__ void load_carried(const Params& p, size_t e, bool mine) {
    load_state(p, e, mine);
    dh_keep = dh;
  }
  static constexpr int kCutInputs = kInputs;
  __device__ __forceinline__ static int cut_input(int i) { return i; }
  __device__ __forceinline__ void carry_inputs(float (&)[kInputs]) {}
};

// The same on the caller's half tensors: h, v, dh_next and zoneout_mask are read, dp and dq written in half.
struct GruHalfScatterCell : GruScatterCell {
  typedef _Float16 half_t;
  __device__ __forceinline__ static void request(const Params& p, float (&in)[kInputs], size_t e, size_t ve,
                                                 bool zoneout) {
    auto half = [](const float* q) { return reinterpret_cast<const half_t*>(q); };
    const half_t* vt = half(p.v) + ve;
#pragma unroll
    for (int i = 0; i < 4; ++i) in[i] = (float)vt[i * (size_t)p.H];
    in[4] = (float)half(p.h)[e];
    in[5] = (float)half(p.dh_next)[e];
    if (zoneout) in[6] = (float)half(p.zoneout_mask)[e];
  }
  __device__ __forceinline__ static void store_copy(const Params& p, int t, size_t n, size_t j, const float4_t& a) {
    const size_t H = p.H;
    const size_t o3 = ((size_t)t * p.N + n) * 3 * H + j;
    half_t *dp = reinterpret_cast<half_t*>(p.dp) + o3, *dq = reinterpret_cast<half_t*>(p.dq) + o3;
    const half_t z = (half_t)a[0], r = (half_t)a[1];
    dp[0] = z;
    dp[H] = r;
    dp[2 * H] = (half_t)a[3];
    dq[0] = z;
    dq[H] = r;
    dq[2 * H] = (half_t)a[2];
  }
};

}  // namespace
}  // namespace haste_hip
