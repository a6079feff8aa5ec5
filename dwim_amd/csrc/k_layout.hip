// The device layouts of layout.h made on the device from the host formats as
// they were copied (`Device::upload`, dwim gpu/mod.rs:206): one pass at memory
// speed, a thread a 16-byte chunk, where the host would place 16 bytes at a
// time.
#include "layout.h"
#include "runtime.h"

namespace {

constexpr size_t kTile = rowt::kTile;

// Q4_0 (per = 4) and Q8_0 (per = 8): chunk i of the layout, from row-major chunks
__global__ void k_tile_chunks(uint4 *__restrict__ dst, const uint4 *__restrict__ src, size_t rows, size_t cols,
                              unsigned per, size_t count) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= count) return;
    const size_t units = rowt::units(cols), row = i / kTile / per / units * kTile + i % kTile;
    const size_t j = i / kTile / per % units * per + i / kTile % per;  // the row's chunk
    const size_t in_row = cols / 32 * (per / 4);
    dst[i] = row < rows && j < in_row ? src[row * in_row + j] : make_uint4(0, 0, 0, 0);
}

__global__ void k_tile_scales(uint16_t *__restrict__ dst, const uint16_t *__restrict__ src, size_t rows, size_t cols,
                              size_t count) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= count) return;
    const size_t units = rowt::units(cols), row = i / 4 / kTile / units * kTile + i / 4 % kTile;
    const size_t b = i / 4 / kTile % units * 4 + i % 4, nb = cols / 32;
    dst[i] = row < rows && b < nb ? src[row * nb + b] : (uint16_t)0;
}

// ggml's block_q6_K, 210 bytes (ql[128], qh[64], sc[16], d): a thread a chunk,
// 14 a block (8 of ql, 4 of qh, sc, d)
__global__ void k_tile_q6k(uint4 *__restrict__ ql, uint4 *__restrict__ qh, uint4 *__restrict__ sc,
                           uint16_t *__restrict__ d, const uint8_t *__restrict__ src, size_t rows, size_t nb,
                           size_t count) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= count) return;
    const size_t blk = i / 14, k = i % 14, row = blk / nb, b = blk % nb;
    const bool in = row < rows;
    const uint8_t *p = src + (in ? blk * 210 + 16 * k : 0);
    if (k == 13) {
        d[rowt::q6_row(nb, row, b)] = in ? (uint16_t)(p[0] | p[1] << 8) : (uint16_t)0;
        return;
    }
    uint32_t v[4];
#pragma unroll
    for (int w = 0; w < 4; w++) {  // (blocks start on even bytes)
        const uint16_t *h = (const uint16_t *)(p + 4 * w);
        v[w] = in ? h[0] | (uint32_t)h[1] << 16 : 0u;
    }
    const uint4 q = make_uint4(v[0], v[1], v[2], v[3]);
    if (k < 8) ql[rowt::ql_chunk(nb, row, b, k)] = q;
    else if (k < 12) qh[rowt::qh_chunk(nb, row, b, k - 8)] = q;
    else sc[rowt::q6_row(nb, row, b)] = q;
}

unsigned blocks_of(size_t count) { return (unsigned)((count + 255) / 256); }

}  // namespace

hipError_t launch_tile_q4_0(hipStream_t s, void *q, const void *src, size_t rows, size_t cols) {
    const size_t n = rowt::chunks(rows, cols, 4);
    k_tile_chunks<<<blocks_of(n), 256, 0, s>>>((uint4 *)q, (const uint4 *)src, rows, cols, 4, n);
    return hipGetLastError();
}

hipError_t launch_tile_q8_0(hipStream_t s, void *q, const void *src, size_t rows, size_t cols) {
    const size_t n = rowt::chunks(rows, cols, 8);
    k_tile_chunks<<<blocks_of(n), 256, 0, s>>>((uint4 *)q, (const uint4 *)src, rows, cols, 8, n);
    return hipGetLastError();
}

hipError_t launch_tile_scales(hipStream_t s, void *scales, const void *src, size_t rows, size_t cols) {
    const size_t n = rowt::scales(rows, cols);
    k_tile_scales<<<blocks_of(n), 256, 0, s>>>((uint16_t *)scales, (const uint16_t *)src, rows, cols, n);
    return hipGetLastError();
}

hipError_t launch_tile_q6_k(hipStream_t s, void *ql, void *qh, void *sc, void *d, const void *src, size_t rows,
                            size_t cols) {
    const size_t nb = cols / 256, n = rowt::tiles(rows) * kTile * nb * 14;
    k_tile_q6k<<<blocks_of(n), 256, 0, s>>>((uint4 *)ql, (uint4 *)qh, (uint4 *)sc, (uint16_t *)d, (const uint8_t *)src,
                                            rows, nb, n);
    return hipGetLastError();
}
