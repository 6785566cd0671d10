// GEMM kernel instances for many activation rows (every alpha format).
#include "lut_gemm_tile_device.h"
#include "lutgemm_launch.h"

namespace lutgemm {
namespace {

template <int NB, int FMT>
hipError_t launch_fmt(const TileProblem &p, hipStream_t stream)
{
    const dim3 grid((unsigned)((p.n_tiles * p.ksplit + 7) / 8 * 8 * p.m_tiles)), block(kTileThreads);
    if (p.tile_rows == 64)
        hipLaunchKernelGGL((lut_gemm_tile_kernel<NB, FMT, 2>), grid, block, 0, stream, p);
    else
        hipLaunchKernelGGL((lut_gemm_tile_kernel<NB, FMT, 4>), grid, block, 0, stream, p);
    return hipGetLastError();
}

template <int NB>
hipError_t launch_nb(const TileProblem &p, hipStream_t stream)
{
    if (p.mode == kRowF16) return launch_fmt<NB, kTileRow>(p, stream);
    if (p.mode == kUniformF16) return launch_fmt<NB, kTileUniform>(p, stream);
    if (p.rows_per_group % kTileWaveN == 0) return launch_fmt<NB, kTileBlockWide>(p, stream);
    return launch_fmt<NB, kTileBlock>(p, stream);
}

}  // namespace

hipError_t launch_tile(const TileProblem &p, int nb, hipStream_t stream)
{
    if (p.ksplit > 1 && !p.partial) return launch_tile_serial(p, nb, stream);
    hipError_t e = hipSuccess;
    if (p.pair)
        e = launch_tile_pair(p, nb, stream);
    else if (nb == 1)
        e = launch_nb<1>(p, stream);
    else if (nb == 2)
        e = launch_nb<2>(p, stream);
    else if (nb == 3)
        e = launch_nb<3>(p, stream);
    else
        e = launch_nb<4>(p, stream);
    if (p.ksplit == 1 || e != hipSuccess) return e;
    hipLaunchKernelGGL(tile_sum_kernel, dim3((unsigned)(((size_t)p.M * p.N / 4 + 255) / 256)), dim3(256), 0, stream, p);
    return hipGetLastError();
}

}  // namespace lutgemm
