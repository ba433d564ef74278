// transfer_kernels.h -- layout and precision conversion between the dense
// FP64 arrays of the ABI (rows of nx values) and the plan's padded rows
// (pitch px, plan precision), on the device.
//
// A host copy of a padded array row by row (hipMemcpy2D to or from pageable
// memory) costs about 7 us per row whatever the row's length: 631 ms for the
// 88,804 rows of a 298^3 FP64 field, 0.3 GB/s.  Packing on the device leaves
// one contiguous copy, which the runtime moves at 10 (pages touched for the
// first time) to 28 GB/s: 20 ms for the same field.  The kernels themselves
// stream at HBM rate and are a hundredth of the copy.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "stencil_kernels.h"  // kTileX

namespace awcpml {

constexpr int kRowSeg = 1024;  // elements of one row a block converts at a time

// dst[r*dpitch + i] = src[r*spitch + i] for i < nx, r < rows.  A block takes
// segments of kRowSeg elements, so that one long row (traces, wavelets)
// spreads over the chip as well as many short ones do.
template <typename S, typename D>
__global__ __launch_bounds__(256) void convert_rows(const S* src, D* dst, int64_t nx, int64_t spitch,
                                                    int64_t dpitch, int64_t rows) {
    const int64_t segs = (nx + kRowSeg - 1) / kRowSeg;
    for (int64_t u = blockIdx.x; u < segs * rows; u += gridDim.x) {
        const int64_t r = u / segs, i0 = (u - r * segs) * kRowSeg;
        for (int i = (int)threadIdx.x; i < kRowSeg && i0 + i < nx; i += 256)
            dst[r * dpitch + i0 + i] = (D)src[r * spitch + i0 + i];
    }
}

// The aligned two-step tiles' edge copy of fact (x = 64*t-1 and 64*t+64,
// clamped into the interior): 3D [z][t][side][y], 2D [y][t][side].
template <typename T>
__global__ __launch_bounds__(256) void gather_fact_edge(const T* fact, T* edge, int64_t nx, int64_t px,
                                                        int64_t ny, int64_t tiles, int three_d,
                                                        int64_t count) {
    for (int64_t q = (int64_t)blockIdx.x * 256 + threadIdx.x; q < count; q += (int64_t)gridDim.x * 256) {
        const int64_t j = three_d ? q % ny : 0, e = three_d ? q / ny : q;
        const int64_t k = e / 2 / tiles, t = e / 2 % tiles;
        int64_t x = e % 2 == 0 ? t * kTileX - 1 : t * kTileX + kTileX;
        x = x < 1 ? 1 : (x > nx - 2 ? nx - 2 : x);
        edge[q] = fact[x + px * (j + (three_d ? ny : 1) * k)];
    }
}

// Several buffers copied in one launch: a checkpoint of the forward run is up to
// 15 of them.  Small ones cost their launch (4.6 us each with hipMemcpyAsync;
// 81x73x69 FP64, 2 shots: 69 us per checkpoint, 14 so), large ones run at HBM rate
// either way.  Buffers are 16-byte aligned; sizes are multiples of 4 bytes.
constexpr int kMaxPieces = 15;
struct CopyPieces {
    const void* src[kMaxPieces];
    void* dst[kMaxPieces];
    uint64_t bytes[kMaxPieces];
    int count;
};

static __global__ __launch_bounds__(256) void copy_pieces(const CopyPieces P) {
    const uint64_t first = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (int q = 0; q < P.count; ++q) {
        const uint64_t n16 = P.bytes[q] / 16, n4 = P.bytes[q] / 4;
        for (uint64_t u = first; u < n16; u += stride) ((uint4*)P.dst[q])[u] = ((const uint4*)P.src[q])[u];
        for (uint64_t u = n16 * 4 + first; u < n4; u += stride)
            ((uint32_t*)P.dst[q])[u] = ((const uint32_t*)P.src[q])[u];
    }
}

}  // namespace awcpml
