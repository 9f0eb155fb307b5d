// Rows of 16-bit elements at any alignment as the 16-byte operand pieces of the matrix kernels.
#pragma once
#include "ba_gemm_common.hpp"

namespace ba {

constexpr uint32_t kNowhere = 0xfffffff0u;            // byte offset no segment reaches

// Rows of K elements read as 16-byte pieces (eight elements from column 8 p on) through a buffer descriptor that spans
// the segment.  VEC: K is a multiple of 8, every piece lies inside a row, rows past the last read as zeros.  Otherwise a
// piece may reach past its row's end (those elements are cleared) and the last ones past the segment's end: they are
// read from the last 16 bytes of the segment and shifted down.  A segment of fewer than eight elements is read element by element.
template <bool VEC> struct RowPieces {
    __amdgpu_buffer_rsrc_t res;
    uint32_t bytes, row_bytes;
    int K;
    __device__ __forceinline__ RowPieces(const uint16_t *seg, int rows, int K_) {
        K = K_;
        row_bytes = 2u * (uint32_t)K_;
        bytes = (uint32_t)rows * row_bytes;
        res = __builtin_amdgcn_make_buffer_rsrc((void *)seg, 0, bytes, kRsrcFlags);
    }
    __device__ __forceinline__ uint32_t offset(int row, int piece) const {
        return 8 * piece < K ? (uint32_t)row * row_bytes + 16u * (uint32_t)piece : kNowhere;
    }
    __device__ __forceinline__ u32x4 load(uint32_t off) const {
        if constexpr (VEC) return __builtin_amdgcn_raw_buffer_load_b128(res, off, 0, 0);
        if (bytes >= 16) return __builtin_amdgcn_raw_buffer_load_b128(res, min(off, bytes - 16), 0, 0);
        u32x4 x = {0u, 0u, 0u, 0u};
#pragma nounroll
        for (int i = 0; i < 8; ++i) {                 // each step shifts the piece down and puts an element on top
            const uint32_t e = __builtin_amdgcn_raw_buffer_load_b16(res, off + 2 * i, 0, 0);
            x = u32x4{__builtin_amdgcn_alignbit(x[1], x[0], 16), __builtin_amdgcn_alignbit(x[2], x[1], 16),
                      __builtin_amdgcn_alignbit(x[3], x[2], 16), (x[3] >> 16) | (e << 16)};
        }
        return x;
    }
    // what load(off) returned -> the piece (no-op for VEC)
    __device__ __forceinline__ u32x4 finish(u32x4 x, uint32_t off, int piece) const {
        if constexpr (VEC) return x;
        if (bytes >= 16) {
            // (elements 0 .. 8; a piece past the row's end is cleared below: shifting those too would run for every block of a
            // head dimension with lanes to spare, 16 x 4 pairs of 1000 .. 2000 rows, K = 101: forward 187 -> 159 us, backward 423 -> 378)
            const uint32_t behind = 8 * piece >= K || off <= bytes - 16 ? 0u : (min(off, bytes) - (bytes - 16)) >> 1;
            if (__any(behind != 0)) {
                if (behind & 8) x = u32x4{0u, 0u, 0u, 0u};
                if (behind & 4) x = u32x4{x[2], x[3], 0u, 0u};
                if (behind & 2) x = u32x4{x[1], x[2], x[3], 0u};
                if (behind & 1)
                    x = u32x4{__builtin_amdgcn_alignbit(x[1], x[0], 16), __builtin_amdgcn_alignbit(x[2], x[1], 16),
                              __builtin_amdgcn_alignbit(x[3], x[2], 16), x[3] >> 16};
            }
        }
        const int left = K - 8 * piece;               // elements of the row from this piece on
        if (left < 8) {
#pragma unroll
            for (int w = 0; w < 4; ++w) x[w] &= left >= 2 * w + 2 ? 0xffffffffu : left == 2 * w + 1 ? 0xffffu : 0u;
        }
        return x;
    }
    __device__ __forceinline__ u32x4 get(int row, int piece) const {
        const uint32_t off = offset(row, piece);
        return finish(load(off), off, piece);
    }
};

}  // namespace ba
