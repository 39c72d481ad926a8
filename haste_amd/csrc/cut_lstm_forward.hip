// The LSTM's forward recurrence on several XCDs (cut_recurrence.h).
#include "cut_recurrence.h"
#include "lstm_cells.h"

namespace haste_hip {

int lstm_forward_cut(hipStream_t stream, int training, int T, int N, int C, int H, const float* W, const float* R,
                     const float* b, const float* x, const float* h, const float* c, float* h_out, float* c_out, float* v,
                     float zoneout_prob, const float* zoneout_mask, const float* dc_mask, float dc_scale, const CutOther& other, bool* taken) {
  CutPlan cut;
  HASTE_HIP_PROPAGATE((cut_rule<LstmForwardCell, false>(stream, T, N, H, other, dc_mask != nullptr, &cut)));
  *taken = cut.ok;
  if (!cut.ok) return HASTE_HIP_OK;
  HASTE_HIP_PROPAGATE(gemm_f32(stream, false, T * N, 4 * H, C, x, C, W, 4 * H, v, 4 * H, false));
  LstmFwdParams p{};
  p.training = training; p.T = T; p.N = N; p.H = H;
  p.R = R; p.b = b; p.h = h; p.c = c; p.h_out = h_out; p.c_out = c_out; p.v = v;
  p.zoneout_prob = zoneout_prob; p.zoneout_mask = zoneout_mask;
  p.dc_mask = dc_mask; p.dc_scale = dc_scale;
  return launch_cut<LstmForwardCell, false>("lstm_forward_recurrence", stream, cut, p);
}

}  // namespace haste_hip
