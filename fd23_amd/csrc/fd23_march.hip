// Instances of the marching kernels (a translation unit of its own: each
// holds three or six unrolled row loops).
#include "fd23.h"
#include "fd_march.hpp"
#include "fd_sh_march.hpp"

namespace fd23 {

template <class S>
void march_launch(hipStream_t stream, const PsvFields<S> &fa, const PsvFields<S> &fb, const PsvMat5<float> &m,
                  const Grid &g, const MarchWork &w, const FusedEvents &ev, const float *sa, const float *scl,
                  unsigned *amax) {
    const dim3 grid((w.nwork + 7) / 8 * 8), block(w.W / NC);
    if (w.W == 256)
        hipLaunchKernelGGL((k_psv_march<S, 256>), grid, block, 0, stream, fa, fb, m, g, w, ev, sa, scl, amax);
    else
        hipLaunchKernelGGL((k_psv_march<S, 512>), grid, block, 0, stream, fa, fb, m, g, w, ev, sa, scl, amax);
}

#define INSTANCE(S)                                                                                                  \
    template void march_launch<S>(hipStream_t, const PsvFields<S> &, const PsvFields<S> &, const PsvMat5<float> &,   \
                                  const Grid &, const MarchWork &, const FusedEvents &, const float *, const float *, \
                                  unsigned *);
INSTANCE(float)
INSTANCE(__half)
INSTANCE(__hip_bfloat16)
#undef INSTANCE

void sh_march_launch(hipStream_t stream, const ShFields<float> &fa, const ShFields<float> &fb, const ShMat3<float> &m,
                     const Grid &g, const MarchWork &w, const FusedEvents &ev) {
    const dim3 grid((w.nwork + 7) / 8 * 8), block(w.W / NC);
    if (w.W == 256) hipLaunchKernelGGL((k_sh_march<256>), grid, block, 0, stream, fa, fb, m, g, w, ev);
    else hipLaunchKernelGGL((k_sh_march<512>), grid, block, 0, stream, fa, fb, m, g, w, ev);
}

} // namespace fd23
