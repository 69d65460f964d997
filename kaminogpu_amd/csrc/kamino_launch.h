// kamino_launch.h -- host launchers of the step kernels (kamino_kernels.hip).
#pragma once

#include <hip/hip_runtime.h>

#include "kamino_device.h"

namespace kam {

// An advection tile of R rows and W <= 128 columns stages its input fields
// over R + 2 kAdvHaloRows rows and W + 2 kAdvHaloCols columns of LDS, at a
// row stride of adv_stride(W) floats (W rounded up to 64 or 128, plus halo).
constexpr int kAdvHaloRows = 3, kAdvHaloCols = 4, kAdvMaxCols = 128, kAdvMaxRows = 64;
constexpr int adv_stride(int W) { return (W <= 64 ? 64 : 128) + 2 * kAdvHaloCols; }

// LDS row stride, in complex values, of a row of M in the row FFT.  Four past
// its end, so that the rows of a tile start in different banks (the spectrum
// is read and written across them); with `padded` (the kernels of one
// power-of-two size) one slot is left free after every 16 values too.
constexpr int fft_row_stride(int M, bool padded) { return M + (padded ? M >> 4 : 0) + 4; }

// polarD: columns that polar tiles stage on either side of theirs (PolarStage),
// a multiple of 4, at most half of every member's nPhi.
// waves: wavefronts of a workgroup, kAdvWaves or, at the narrower stride,
// kAdvWavesWide.
constexpr int kAdvWaves = 4, kAdvWavesWide = 8;
hipError_t launch_advect(const SimDesc* sims, const Tile* tiles, int ntiles, int parity,
                         int stride, int waves, int polarD, size_t ldsBytes, int gridCap, hipStream_t st);
// the first `staged` tiles (at most kPartStaged particles each) sample the
// velocities from LDS, ldsBytes of it; the others (at most kPartTile) from
// memory, kPartTile / kPartBlock workgroups to a tile
constexpr int kPartStaged = 8192, kPartTile = 2048, kPartBlock = 256;
hipError_t launch_particles(const SimDesc* sims, const Tile* tiles, int ntiles, int staged, size_t ldsBytes,
                            int parity, int gridCap, hipStream_t st);
// kernel: M where every row FFT of the launch has the same length M = 2^k >= 32
// (FftPow2); else 1 when some rows span wavefronts, 0 when none does.
hipError_t launch_div_fft(const SimDesc* sims, const Tile* tiles, int ntiles, int parity,
                          size_t ldsBytes, int gridCap, hipStream_t st, int kernel);
// `parity` names the current state copy: a simulation with the FP64 pressure
// keeps its solved spectrum over the other one.
// fp32: run the elimination in FP32 with subtraction-free pivots (the FP32
// pressure); else in FP64 (the FP64 pressure).
hipError_t launch_tridiag(int lanesPerMode, int kmax, const SimDesc* sims, const Tile* tiles,
                          int ntiles, int parity, int gridCap, hipStream_t st, bool resid = false,
                          bool fp32 = false);
// p64: the tiles belong to simulations with the FP64 pressure (SIM_P64).
// pout (one simulation only): write its pressure rows there instead of
// updating the velocities.
hipError_t launch_ifft_grad(const SimDesc* sims, const Tile* tiles, int ntiles, int parity,
                            size_t ldsBytes, int gridCap, hipStream_t st, int kernel, bool p64 = false,
                            float* pout = nullptr);

// The phi transforms of SIM_DFT simulations (kamino_dft.hip): divergence rows
// + forward DFT product, and inverse DFT product + gradient rows.  rowTiles
// are row runs of the simulations, gemmTiles 64-row x 128-column output
// blocks (row0, rows, col0).
hipError_t launch_dft_forward(const SimDesc* sims, const Tile* rowTiles, int nRow, const Tile* gemmTiles,
                              int nGemm, int parity, hipStream_t st);
hipError_t launch_dft_inverse(const SimDesc* sims, const Tile* rowTiles, int nRow, const Tile* gemmTiles,
                              int nGemm, int parity, hipStream_t st);
// The inverse DFT product alone: pressure rows over the finished state copy.
hipError_t launch_dft_pressure(const SimDesc* sims, const Tile* gemmTiles, int nGemm, int parity,
                               hipStream_t st);
constexpr int kDftTileRows = 64, kDftTileCols = 128, kDftChunk = 32;

// Ranges of 4-byte values to copy (src given) or to clear (src null) by one
// launch; the kernel reads and writes them, so they are this device's memory or
// pinned host memory.  A runtime copy between pinned and device memory goes to a
// copy engine and back, 10 us and more in the stream for a few kilobytes: with
// an engine's tables and finished fields moved by this kernel, 40 steps of 96
// spheres of 32 to 512 rows with twelve retirements take 8.4 ms instead of 9.2
// (48 steps of 64 spheres of 32 to 256 rows with eight: 4.0 to 4.6 and 4.4 to
// 4.8).  A copy stream beside the engine's for the finished fields: the same.
constexpr int kMaxRanges = 6;
struct Ranges {
    void* dst[kMaxRanges];
    const void* src[kMaxRanges];
    int64_t n[kMaxRanges];  // values
};
hipError_t launch_ranges(const Ranges& a, hipStream_t st);

// Raises the dynamic-LDS limit of every step kernel to `bytes` (call once).
hipError_t configure_kernels(size_t bytes);

}  // namespace kam
