// Matrix-core kernel instances (a few activation rows, every alpha format).
#include "lut_gemm_mfma_device.h"
#include "lutgemm_launch.h"

namespace lutgemm {
namespace {

template <int NB, int FMT, bool OWN>
hipError_t launch_fmt(const Problem &p, int mt, hipStream_t stream)
{
    const dim3 grid((unsigned)p.n_blocks), block(kMfmaThreads);
    const bool one = p.sets_per_split == kMfmaWaves;  // one round per K-slice
    if (mt == 2 && one)
        hipLaunchKernelGGL((lut_gemm_mfma_kernel<NB, 2, FMT, OWN, true>), grid, block, 0, stream, p);
    else if (mt == 2)
        hipLaunchKernelGGL((lut_gemm_mfma_kernel<NB, 2, FMT, OWN, false>), grid, block, 0, stream, p);
    else if (one)
        hipLaunchKernelGGL((lut_gemm_mfma_kernel<NB, 1, FMT, OWN, true>), grid, block, 0, stream, p);
    else
        hipLaunchKernelGGL((lut_gemm_mfma_kernel<NB, 1, FMT, OWN, false>), grid, block, 0, stream, p);
    return hipGetLastError();
}

template <int NB>
hipError_t launch_nb(const Problem &p, int mt, hipStream_t stream)
{
    // tables shared by the wave need steps of 128 inputs inside one alpha group
    const bool own = p.K % kMfmaStepK != 0 || p.group_words % 4 != 0;
    if (p.alpha_mode == kRowF16)
        return own ? launch_fmt<NB, kWeightRow, true>(p, mt, stream) : launch_fmt<NB, kWeightRow, false>(p, mt, stream);
    if (p.alpha_mode == kUniformF16)
        return own ? launch_fmt<NB, kWeightUniform, true>(p, mt, stream) : launch_fmt<NB, kWeightUniform, false>(p, mt, stream);
    return launch_fmt<NB, kWeightBlock, false>(p, mt, stream);
}

template <int NB>
hipError_t launch_fused_nb(const Problem &p, int mt, hipStream_t stream)
{
    const dim3 grid((unsigned)p.n_blocks), block(kMfmaThreads);
    if (mt == 1 && p.sets_per_split == kMfmaWaves)  // one round per K-slice
        hipLaunchKernelGGL((lut_gemm_mfma_fused_kernel<NB, 1, true>), grid, block, 0, stream, p);
    else if (mt == 2)
        hipLaunchKernelGGL((lut_gemm_mfma_fused_kernel<NB, 2>), grid, block, 0, stream, p);
    else
        hipLaunchKernelGGL((lut_gemm_mfma_fused_kernel<NB, 1>), grid, block, 0, stream, p);
    return hipGetLastError();
}

}  // namespace

hipError_t launch_mfma_fused(const Problem &p, int mt, hipStream_t stream)
{
    switch (p.nb) {
    case 1: return launch_fused_nb<1>(p, mt, stream);
    case 2: return launch_fused_nb<2>(p, mt, stream);
    case 3: return launch_fused_nb<3>(p, mt, stream);
    default: return launch_fused_nb<4>(p, mt, stream);
    }
}

hipError_t launch_mfma(const Problem &p, int mt, hipStream_t stream)
{
    switch (p.nb) {
    case 1: return launch_nb<1>(p, mt, stream);
    case 2: return launch_nb<2>(p, mt, stream);
    case 3: return launch_nb<3>(p, mt, stream);
    default: return launch_nb<4>(p, mt, stream);
    }
}

hipError_t launch_mfma_group(const Group &g, int mt, int blocks, hipStream_t stream)
{
    const dim3 grid((unsigned)blocks, (unsigned)g.count), block(kMfmaThreads);
    if (mt == 2)
        hipLaunchKernelGGL((lut_gemm_mfma_group_kernel<2>), grid, block, 0, stream, g);
    else
        hipLaunchKernelGGL((lut_gemm_mfma_group_kernel<1>), grid, block, 0, stream, g);
    return hipGetLastError();
}

hipError_t launch_mfma_gated(const GatedProblems &g, int mt, int blocks, hipStream_t stream)
{
    const dim3 grid((unsigned)blocks, 2u), block(kMfmaThreads);
    if (mt == 2)
        hipLaunchKernelGGL((lut_gemm_mfma_gated_kernel<2>), grid, block, 0, stream, g);
    else
        hipLaunchKernelGGL((lut_gemm_mfma_gated_kernel<1>), grid, block, 0, stream, g);
    return hipGetLastError();
}

}  // namespace lutgemm
