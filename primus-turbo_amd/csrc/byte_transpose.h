// 128 x 128 byte-transpose tile shared by the dense and the grouped byte
// transposes (fp8 operands moved to K-contiguous form).
//
// Bound by memory: every byte is read once and written once.  A 256-thread
// workgroup takes a 128 x 128 tile; each lane loads 16 columns of 4 consecutive
// rows (8 lanes cover a row's 128 bytes), transposes 4 x 4 byte blocks in
// registers (8 v_perm each) so that a dword holds 4 rows of one column, and the
// tile passes through LDS as dwords.  The LDS dword index is XORed with the
// column group, so the writes put 2 lanes on a bank (the least for 64 lanes) and
// the 16-byte reads of the output rows are conflict-free.
#pragma once
#include "common.h"

namespace pta {

constexpr int BT_TILE = 128;
constexpr int BT_NT   = 256;

// out[c] = bytes (r0.c, r1.c, r2.c, r3.c)
__device__ __forceinline__ void byte_transpose4(uint32_t r0, uint32_t r1, uint32_t r2, uint32_t r3, uint32_t (&o)[4]) {
    const uint32_t t0 = __builtin_amdgcn_perm(r1, r0, 0x05010400u), t1 = __builtin_amdgcn_perm(r1, r0, 0x07030602u);
    const uint32_t u0 = __builtin_amdgcn_perm(r3, r2, 0x05010400u), u1 = __builtin_amdgcn_perm(r3, r2, 0x07030602u);
    o[0] = __builtin_amdgcn_perm(u0, t0, 0x05040100u);
    o[1] = __builtin_amdgcn_perm(u0, t0, 0x07060302u);
    o[2] = __builtin_amdgcn_perm(u1, t1, 0x05040100u);
    o[3] = __builtin_amdgcn_perm(u1, t1, 0x07060302u);
}

// Access width in bytes (16, 8 or 1) that a row stride and a base pointer allow.
inline int bt_access(const void *p, int64_t ld) {
    const uint64_t v = reinterpret_cast<uintptr_t>(p) | static_cast<uint64_t>(ld);
    return v % 16 == 0 ? 16 : (v % 8 == 0 ? 8 : 1);
}

// dst[c * ldd + r] = src[r * lds + c] for c < ncols and r < wrows (both at most
// BT_TILE); source rows r >= vrows read as zero.  G: access width; lds, ldd,
// ncols and wrows are multiples of it, the pointers aligned to it.
template <int G>
__device__ __forceinline__ void byte_transpose_tile(const uint8_t *src, int64_t lds, int vrows, int ncols, uint8_t *dst,
                                                    int64_t ldd, int wrows) {
    __shared__ __attribute__((aligned(16))) uint32_t s[BT_TILE][BT_TILE / 4];
    const int t = threadIdx.x;
    {
        const int cseg = t & 7, rg = t >> 3;
        uint32_t  w[4][4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int      r = 4 * rg + i;
            const uint8_t *p = src + r * lds + cseg * 16;
#pragma unroll
            for (int j = 0; j < 4; ++j) w[i][j] = 0u;
            if (r >= vrows) continue;
            if constexpr (G == 16) {
                if (cseg * 16 < ncols) {
                    const uint4 v = *reinterpret_cast<const uint4 *>(p);
                    w[i][0] = v.x; w[i][1] = v.y; w[i][2] = v.z; w[i][3] = v.w;
                }
            } else if constexpr (G == 8) {
#pragma unroll
                for (int h = 0; h < 2; ++h)
                    if (cseg * 16 + 8 * h < ncols) {
                        const uint2 v = *reinterpret_cast<const uint2 *>(p + 8 * h);
                        w[i][2 * h] = v.x; w[i][2 * h + 1] = v.y;
                    }
            } else {
#pragma unroll
                for (int j = 0; j < 16; ++j)
                    if (cseg * 16 + j < ncols) w[i][j >> 2] |= static_cast<uint32_t>(p[j]) << (8 * (j & 3));
            }
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            uint32_t o[4];
            byte_transpose4(w[0][j], w[1][j], w[2][j], w[3][j], o);
#pragma unroll
            for (int k = 0; k < 4; ++k) s[cseg * 16 + 4 * j + k][rg ^ (cseg << 2)] = o[k];
        }
    }
    __syncthreads();
#pragma unroll
    for (int it = 0; it < 4; ++it) {
        const int c = it * (BT_NT / 8) + (t >> 3), q = t & 7; // output row, its 16-byte chunk
        if (c >= ncols) continue;
        const uint4 v = *reinterpret_cast<const uint4 *>(&s[c][(q ^ ((c >> 4) & 7)) << 2]);
        uint8_t    *p = dst + c * ldd + q * 16;
        if constexpr (G == 16) {
            if (q * 16 < wrows) *reinterpret_cast<uint4 *>(p) = v;
        } else if constexpr (G == 8) {
            if (q * 16 < wrows) *reinterpret_cast<uint2 *>(p) = make_uint2(v.x, v.y);
            if (q * 16 + 8 < wrows) *reinterpret_cast<uint2 *>(p + 8) = make_uint2(v.z, v.w);
        } else {
            const uint32_t vs[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (int j = 0; j < 16; ++j)
                if (q * 16 + j < wrows) p[j] = static_cast<uint8_t>(vs[j >> 2] >> (8 * (j & 3)));
        }
    }
}

} // namespace pta
