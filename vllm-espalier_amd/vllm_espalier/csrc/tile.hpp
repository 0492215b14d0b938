// What the prompt launches share (dense_tile.hip, prompt.hip): the A-fragment order of a prompt's rotated rows, and the
// workgroup that makes it.
#pragma once

#include "dense.hpp"

namespace esp {

constexpr int TILE_FRAG = 512;                  // halves an MFMA operand block (16 rows or columns, 32 k): 64 lanes x 8
constexpr int RED_STRIDE = 132;                 // floats between two rows of the block's sums (banks apart)

typedef __attribute__((address_space(3))) const f16x8* lds_f16x8_ptr;

// Rotated rows: a workgroup takes one matrix, one row group of 16 rows and one 128-chunk ch of K, which fill exactly the
// 4 (row group, step) A blocks of that chunk: a 32-lane half rotates 2 rows (rows past T are zero) into their fragment
// places in shared memory (frag, 4 blocks, complete when the call returns). Returns the (matrix, row group)'s blocks in
// xh, one a step.
__device__ __forceinline__ uint16_t* tile_rot_unit(unsigned unit, const void* __restrict__ x, int x_dtype, int x_stride,
                                                   int T, int K, const uint16_t* suh0, const uint16_t* suh1,
                                                   const uint16_t* suh2, const uint16_t* suh3, uint16_t* __restrict__ xh,
                                                   int RG, uint16_t* frag, int& ch) {
    const int l32 = threadIdx.x & 31, hw = threadIdx.x >> 5;
    const int nb = K >> 7;
    const int rg = (int)((unit / nb) % RG), s = (int)(unit / (nb * RG));
    ch = (int)(unit % nb);
    const uint16_t* suh = s == 0 ? suh0 : s == 1 ? suh1 : s == 2 ? suh2 : suh3;
    // the lane's 4 consecutive k (ch * 128 + 4 l32 ...) are 4 consecutive halves of one A fragment lane
    const int kk = (4 * l32) & 31, kt = kk & 15;
    const int sl = l32 >> 3;                                  // the step inside the chunk
    const int G = 2 * (kk >> 4) + ((kt >> 2) & 1), hi = kt >> 3;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int rr = 2 * hw + i, r = rg * 16 + rr;
        uint2 u = make_uint2(0u, 0u);
        if (r < T) u = rot128(x, x_dtype, (size_t)r * x_stride + ch * 128, suh + ch * 128, l32);
        *reinterpret_cast<uint2*>(frag + (sl * 64 + rr + 16 * G) * 8 + 4 * hi) = u;
    }
    __syncthreads();
    return xh + ((size_t)s * RG + rg) * (K >> 5) * TILE_FRAG;
}

}  // namespace esp
