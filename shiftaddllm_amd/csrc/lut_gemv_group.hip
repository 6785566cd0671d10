// Look-up kernel instances: several row-wise problems per launch, with the fused input
// transforms (none, RMSNorm, SiLU(gate) * x).
#include "lut_gemv_device.h"
#include "lutgemm_launch.h"

namespace lutgemm {

namespace {

template <int XF>
hipError_t launch_xform(const Group &g, int blocks, hipStream_t stream)
{
    const dim3 grid((unsigned)blocks, (unsigned)g.count), block(kThreads);
    bool extra = false;
    for (int i = 0; i < g.count; ++i) extra = extra || g.p[i].next_w || g.p[i].sumsq_out || g.p[i].sumsq_in;
    if (extra)
        hipLaunchKernelGGL((lut_gemv_group_kernel<XF, true>), grid, block, 0, stream, g);
    else
        hipLaunchKernelGGL((lut_gemv_group_kernel<XF, false>), grid, block, 0, stream, g);
    return hipGetLastError();
}

}  // namespace

hipError_t launch_gemv_group(const Group &g, int xform, int blocks, hipStream_t stream)
{
    return xform == kXNorm ? launch_xform<kXNorm>(g, blocks, stream)
           : xform == kXGate ? launch_xform<kXGate>(g, blocks, stream) : launch_xform<kXNone>(g, blocks, stream);
}

}  // namespace lutgemm
