// What runs the recurrence of an LSTM or GRU pass, found by going through the pass's own choices without a launch.
#include "cut_recurrence.h"
#include "gru_cells.h"
#include "lstm_cells.h"

namespace haste_hip {

int lstm_forward_impl(hipStream_t stream, int training, int T, int N, int C, int H, const float* W, const float* R,
                      const float* b, const float* x, const float* h, const float* c, float* h_out, float* c_out, float* v,
                      float zoneout_prob, const float* zoneout_mask, const float* dc_mask, float dc_scale);
int lstm_backward_impl(hipStream_t stream, int T, int N, int C, int H, const float* W_t, const float* R_t,
                       const float* x_t, const float* h, const float* c, const float* c_next, const float* dh_next,
                       const float* dc_next, float* dx, float* dW, float* dR, float* db, float* dh, float* dc, float* v,
                       const float* zoneout_mask);
int gru_forward_impl(hipStream_t stream, int training, int T, int N, int C, int H, const float* W, const float* R,
                     const float* bx, const float* br, const float* x, const float* h, float* h_out, float* v,
                     float* tmp_Wx, float zoneout_prob, const float* zoneout_mask, const float* dc_mask, float dc_scale,
                     bool wx_ready, bool half_product, bool half_io);
int gru_backward_impl(hipStream_t stream, int T, int N, int C, int H, const float* W_t, const float* R_t,
                      const float* x_t, const float* h, const float* v, const float* dh_next, float* dx, float* dW,
                      float* dR, float* dbx, float* dbr, float* dh, float* dp, float* dq, const float* zoneout_mask,
                      bool products, bool half_product, bool half_io);
size_t recurrence64_scratch_bytes(int in_gates, int out_gates, int steps, int N, int H);
int lstm_forward_recurrence64(hipStream_t stream, int training, int T, int N, int H, const double* R, const double* b,
                              const double* h, const double* c, double* h_out, double* c_out, double* v,
                              float zoneout_prob, const double* mask, void* exchange);
int gru_forward_recurrence64(hipStream_t stream, int training, int T, int N, int H, const double* R, const double* bx,
                             const double* br, const double* h, const double* wx, double* h_out, double* v,
                             float zoneout_prob, const double* mask, void* exchange);
int lstm_backward_recurrence64(hipStream_t stream, int T, int N, int H, const double* R_t, const double* c,
                               const double* c_next, const double* dh_next, const double* dc_next, double* dh,
                               double* dc, double* v, const double* mask, void* exchange);
int gru_backward_recurrence64(hipStream_t stream, int T, int N, int H, const double* R_t, const double* h,
                              const double* v, const double* dh_next, double* dh, double* dp, double* dq,
                              const double* mask, void* exchange);

size_t cut_scratch_bound(int N, int H, int cus) {
  size_t most = 0;
  for (int xcds = 1; xcds <= cus; ++xcds) {
    if (cus % xcds != 0) continue;
    auto ask = [&](const CutPlan& plan, size_t weights) {
      if (plan.ok && plan.bytes() + weights > most) most = plan.bytes() + weights;
    };
    const size_t weights = ((size_t)4 * H * H + 64) * sizeof(float);
    ask(cut_plan<LstmForwardCell, false>(N, H, cus, xcds), weights);
    ask(cut_plan<LstmScatterCell, true>(N, H, cus, xcds), 0);
    ask(cut_plan<GruForwardCell, false>(N, H, cus, xcds), weights);
    ask(cut_plan<GruScatterCell, true>(N, H, cus, xcds), 0);
  }
  return most;
}

int plan_recurrence(int gates, int element_bytes, bool backward, int T, int N, int C, int H) {
  const bool lstm = gates == 4;
  if (element_bytes == 8) {
    const size_t bytes = recurrence64_scratch_bytes(backward ? gates : 1, backward ? 1 : gates, T, N, H);
    const size_t lent = planned_pass()->lent;
    if (bytes == 0 || (lent > 0 && lent < bytes)) return HASTE_HIP_OK;  // step by step
    Workspace ws;
    HASTE_HIP_PROPAGATE(get_workspace(nullptr, bytes, &ws));
    double* a = reinterpret_cast<double*>(ws.scratch);  // an address for every tensor: none is read
    if (backward)
      return lstm ? lstm_backward_recurrence64(nullptr, T, N, H, a, a, a, a, a, a, a, a, a, a)
                  : gru_backward_recurrence64(nullptr, T, N, H, a, a, a, a, a, a, a, a, a);
    return lstm ? lstm_forward_recurrence64(nullptr, 1, T, N, H, a, a, a, a, a, a, a, 0.f, nullptr, a)
                : gru_forward_recurrence64(nullptr, 1, T, N, H, a, a, a, a, a, a, a, 0.f, nullptr, a);
  }
  float* a = reinterpret_cast<float*>(uintptr_t(256));
  if (backward)
    return lstm ? lstm_backward_impl(nullptr, T, N, C, H, a, a, a, a, a, a, a, a, a, a, a, a, a, a, a, nullptr)
                : gru_backward_impl(nullptr, T, N, C, H, a, a, a, a, a, a, a, a, a, a, a, a, a, a, nullptr, true, false, false);
  return lstm ? lstm_forward_impl(nullptr, 1, T, N, C, H, a, a, a, a, a, a, a, a, a, 0.f, nullptr, nullptr, 1.f)
              : gru_forward_impl(nullptr, 1, T, N, C, H, a, a, a, a, a, a, a, a, a, 0.f, nullptr, nullptr, 1.f, false, false, false);
}

}  // namespace haste_hip
