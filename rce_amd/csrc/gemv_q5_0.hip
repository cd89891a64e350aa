// gemv_q5_0.hip -- the Q5_0 decode kernels (EXACT and Q8).
#include "qmm_gemv_kernels.h"

namespace rce_qmm {
hipError_t launch_gemv_q5_0(const DevWeight &w, const GemvGeom &g, const float *a, size_t t_rows, float *out, int mode,
                            hipStream_t s) {
    if (mode == 0) return launch_as_tb<Q5_0Exact, false, 4>(w, g, a, t_rows, out, s);
    return launch_as_tb<Q5_0Q8, true, 8>(w, g, a, t_rows, out, s);
}
hipError_t launch_gemv_fx_q5_0(const FxLaunch &f, const GemvGeom &g, const float *a, int mode, hipStream_t s) {
    if (mode == 0) return launch_as_fx_nt<Q5_0Exact<1>, false>(f, g, a, s);
    return launch_as_fx_nt<Q5_0Q8<1>, true>(f, g, a, s);
}
hipError_t launch_gemv_grouped_q5_0(const DevWeight &w, const MoeGroup &m, const void *a, float *out, int mode, hipStream_t s) {
    if (mode == 0) return launch_as_grouped_tb<Q5_0Exact, false>(w, m, a, out, s);
    return launch_as_grouped_tb<Q5_0Q8, true>(w, m, a, out, s);
}
}  // namespace rce_qmm
