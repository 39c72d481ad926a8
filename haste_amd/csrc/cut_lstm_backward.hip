// The LSTM's backward recurrence on several XCDs (cut_recurrence.h).
#include "cut_recurrence.h"
#include "lstm_cells.h"

namespace haste_hip {

int lstm_backward_cut(hipStream_t stream, int T, int N, int H, const float* R_t, const float* c, const float* c_next,
                      const float* dh_next, const float* dc_next, float* db, float* dh, float* dc, float* v,
                      const float* zoneout_mask, const CutOther& other, bool* taken) {
  CutPlan cut;
  HASTE_HIP_PROPAGATE((cut_rule<LstmScatterCell, true>(stream, T, N, H, other, false, &cut)));
  *taken = cut.ok;
  if (!cut.ok) return HASTE_HIP_OK;
  LstmBwdParams p{};
  p.T = T; p.N = N; p.H = H;
  p.R_t = R_t; p.c = c; p.c_next = c_next; p.dh_next = dh_next;
  p.dc_next = dc_next != nullptr ? dc_next : dh_next;
  p.dc_given = dc_next != nullptr;
  p.db = db; p.dh = dh; p.dc = dc; p.v = v; p.zoneout_mask = zoneout_mask;
  return launch_cut<LstmScatterCell, true>("lstm_backward_recurrence", stream, cut, p);
}

}  // namespace haste_hip
