// What the prompt launches share (dense_tile.hip, prompt.hip): the A-fragment order of a prompt's rotated rows, and the
// workgroup that makes it.
#pragma once

#include "dense.hpp"

namespace esp {

constexpr int TILE_FRAG = 512;                  // halves an MFMA operand block (16 rows or columns, 32 k): 64 lanes x 8
constexpr int RED_STRIDE = 132;                 // floats between two rows of the block's sums (banks apart)

typedef __attribute__((address_space(3))) const f16x8* lds_f16x8_ptr;

// Rotated rows: 8 lanes take one (matrix, row, 128-chunk of K) of unit = ((matrix * RG + row group) * K / 128 + chunk) *
// 16 + row of the group (rows past T are zero): a lane's 16 elements are one k-tile's, which two lanes of the chunk's
// step (l8 / 2) hold in halves, 16 bytes each. place(step) is the step's block among the (matrix, row group)'s in xh.
template <typename PLACE>
__device__ __forceinline__ void tile_rot_unit(unsigned unit, const void* __restrict__ x, int x_dtype, int x_stride, int T,
                                              int K, bool wide, const uint16_t* suh0, const uint16_t* suh1,
                                              const uint16_t* suh2, const uint16_t* suh3, uint16_t* __restrict__ xh,
                                              int RG, const PLACE& place) {
    const int lane = threadIdx.x & 63, l8 = lane & 7, nb = K >> 7;
    const int rr = (int)(unit & 15), ch = (int)((unit >> 4) % nb);
    const int rg = (int)((unit >> 4) / nb % RG), s = (int)((unit >> 4) / nb / RG), r = rg * 16 + rr;
    const uint16_t* suh = s == 0 ? suh0 : s == 1 ? suh1 : s == 2 ? suh2 : suh3;
    uint32_t w[8];
    // every lane of the 8 takes the same branch
    if (r < T) {
        rot128_16<16>(x, x_dtype, (size_t)r * x_stride + ch * 128, suh + ch * 128, wide, lane, w);
    } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) w[i] = 0u;
    }
    uint16_t* dst = xh + (((size_t)s * RG + rg) * (K >> 5) + place(ch * 4 + (l8 >> 1))) * TILE_FRAG;
    const int G = 2 * (l8 & 1);                      // the fragment lanes rr + 16 G (k 0-3, 8-11) and G + 1 (4-7, 12-15)
    *reinterpret_cast<uint4*>(dst + (rr + 16 * G) * 8) = make_uint4(w[0], w[1], w[4], w[5]);
    *reinterpret_cast<uint4*>(dst + (rr + 16 * (G + 1)) * 8) = make_uint4(w[2], w[3], w[6], w[7]);
}

constexpr int ROT_UNITS = 32;                        // units a workgroup of 256

// whether rot128_16 may read x and the signs 16 bytes at a time
inline bool rot_wide(const void* x, int64_t x_stride, const uint16_t* const* suh, int n) {
    bool wide = (uintptr_t)x % 16 == 0 && x_stride % 8 == 0;
    for (int i = 0; i < n; ++i) wide = wide && (uintptr_t)suh[i] % 16 == 0;
    return wide;
}

}  // namespace esp
