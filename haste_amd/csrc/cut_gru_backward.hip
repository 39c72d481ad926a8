// The GRU's backward recurrence on several XCDs (cut_recurrence.h).
#include "cut_recurrence.h"
#include "gru_cells.h"

namespace haste_hip {

int gru_backward_cut(hipStream_t stream, int T, int N, int H, const float* R_t, const float* h, const float* v,
                     const float* dh_next, float* dbx, float* dbr, float* dh, float* dp, float* dq,
                     const float* zoneout_mask, const CutOther& other, bool* taken) {
  CutPlan cut;
  HASTE_HIP_PROPAGATE((cut_rule<GruScatterCell, true>(stream, T, N, H, other, false, &cut)));
  *taken = cut.ok;
  if (!cut.ok) return HASTE_HIP_OK;
  GruBwdParams p{};
  p.T = T; p.N = N; p.H = H;
  p.R_t = R_t; p.h = h; p.v = v; p.dh_next = dh_next;
  p.dbx = dbx; p.dbr = dbr; p.dh = dh; p.dp = dp; p.dq = dq; p.zoneout_mask = zoneout_mask;
  return launch_cut<GruScatterCell, true>("gru_backward_recurrence", stream, cut, p);
}

}  // namespace haste_hip
