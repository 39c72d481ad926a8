// The GRU's forward recurrence on several XCDs (cut_recurrence.h).
#include "cut_recurrence.h"
#include "gru_cells.h"

namespace haste_hip {

int gru_forward_cut(hipStream_t stream, int training, int T, int N, int C, int H, const float* W, const float* R,
                    const float* bx, const float* br, const float* x, const float* h, float* h_out, float* v,
                    float* tmp_Wx, float zoneout_prob, const float* zoneout_mask, const float* dc_mask, float dc_scale,
                    bool wx_ready, const CutOther& other, bool* taken) {
  CutPlan cut;
  HASTE_HIP_PROPAGATE((cut_rule<GruForwardCell, false>(stream, T, N, H, other, dc_mask != nullptr, &cut)));
  *taken = cut.ok;
  if (!cut.ok) return HASTE_HIP_OK;
  if (!wx_ready) HASTE_HIP_PROPAGATE(gemm_f32(stream, false, T * N, 3 * H, C, x, C, W, 3 * H, tmp_Wx, 3 * H, false));
  GruFwdParams p{};
  p.training = training; p.T = T; p.N = N; p.H = H;
  p.R = R; p.bx = bx; p.br = br; p.h = h; p.h_out = h_out; p.v = v; p.Wx = tmp_Wx;
  p.zoneout_prob = zoneout_prob; p.zoneout_mask = zoneout_mask;
  p.dc_mask = dc_mask; p.dc_scale = dc_scale;
  return launch_cut<GruForwardCell, false>("gru_forward_recurrence", stream, cut, p);
}

}  // namespace haste_hip
