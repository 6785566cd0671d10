// GEMM kernel instances whose workgroups take the K-slices of a tile in turn (every alpha format).
#include "lut_gemm_tile_device.h"
#include "lutgemm_launch.h"

namespace lutgemm {
namespace {

template <int NB, int FMT>
hipError_t launch_fmt(const TileProblem &p, hipStream_t stream)
{
    const dim3 grid((unsigned)((p.n_tiles + 7) / 8 * 8 * p.m_tiles)), block(kTileThreads);
    if (p.pair)
        hipLaunchKernelGGL((lut_gemm_tile_serial_kernel<NB, FMT, 2, kTileSerialPair>), grid, block, 0, stream, p);
    else if (p.tile_rows == 64)
        hipLaunchKernelGGL((lut_gemm_tile_serial_kernel<NB, FMT, 2, kTileSerial>), grid, block, 0, stream, p);
    else
        hipLaunchKernelGGL((lut_gemm_tile_serial_kernel<NB, FMT, 4, kTileSerial>), grid, block, 0, stream, p);
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

hipError_t launch_tile_serial(const TileProblem &as_planned, int nb, hipStream_t stream)
{
    TileProblem p = as_planned;
    if (p.pair) {   // (the rows of a tile do not matter to the bits; at most 256 tiles of 64 rows, as plan_tile cuts for teams)
        p.tile_rows = 64;
        p.m_tiles = (p.M + 63) / 64;
    }
    switch (nb) {
    case 1: return launch_nb<1>(p, stream);
    case 2: return launch_nb<2>(p, stream);
    case 3: return launch_nb<3>(p, stream);
    default: return launch_nb<4>(p, stream);
    }
}

}  // namespace lutgemm
