// Where the GEMM kernels' buffer loads read, as functions that the kernels and the
// host-side check (pta_test_gemm_stray_reads) share.
//
// A buffer load drops lanes past the descriptor's records.  Whether that check
// compares the lane's offset alone, its sum with the scalar offset, or the lane's
// offset with the records minus the scalar offset (which may wrap) is not relied
// on: every lane either reads inside the operand, or is past the records with a
// scalar offset inside them, where the readings agree.
#pragma once
#include <cstdint>

#include <hip/hip_runtime.h>

namespace pta {
namespace gemm_detail {

#define PTA_HD __host__ __device__ __forceinline__

constexpr int BM = 256, BK = 128;
constexpr int BN = 256;             // default tile width (128 for tail tiles)
constexpr int HALF = 128;           // rows of an operand tile's half (one LDS item)
constexpr int OOB_LANE = 0x7fffffff - 64; // a lane offset past every descriptor's records

PTA_HD int32_t desc_records(int64_t bytes) { return bytes > 0x7fffffff ? 0x7fffffff : static_cast<int32_t>(bytes); }

// First row and row count of half h of an operand tile, `rows` being left from the
// tile's first on (at least one).  A half without rows stands for the tile's first row:
// its loads stay inside the operand, and nothing of what they bring is stored.
PTA_HD int half_start(int64_t rows, int h) { return rows > HALF * h ? HALF * h : 0; }
PTA_HD int half_rows(int64_t rows, int h) {
    const int64_t r = rows - HALF * h;
    return r <= 0 ? 1 : (r < HALF ? static_cast<int>(r) : HALF);
}

// Bytes from a half's first row to the end of its last row's K bytes.
PTA_HD int64_t half_bytes(int rows, int64_t ld, int64_t K) { return (rows - 1) * ld + K; }

// Lane offset of a half's row r, 16-byte chunk ch of a K block.
PTA_HD int lane_off(int r, int64_t ld, int ch) { return r * static_cast<int>(ld) + 16 * ch; }

// The K block that K cuts (none: larger than any), and whether chunk ch of it lies past
// K: those lanes take OOB_LANE.
PTA_HD int  cut_block(int nk, int64_t K) { return (K % BK) != 0 ? nk - 1 : 0x7fffffff; }
PTA_HD bool past_k(int nk, int64_t K, int ch) { return (nk - 1) * BK + 16 * ch >= K; }

// Scalar offset and records of K block kb: none past the last.
PTA_HD int item_soff(int kb, int nk) { return kb < nk ? kb * BK : 0; }
PTA_HD int item_records(int records, int kb, int nk) { return kb < nk ? records : 0; }

// Lane offset of row r's scales, in elements of `es` bytes (two_d: one row of scales per
// 128 rows).
PTA_HD int scale_off(int64_t r, bool two_d, int64_t stride, int es) {
    return static_cast<int>((two_d ? (r >> 7) : r) * stride) * es;
}

// Row whose scales a lane reads for row r: rows past the end read the last row's.
PTA_HD int64_t scale_row(int64_t r, int64_t rows) { return r < rows ? r : rows - 1; }

// K block whose scales a load for block kb reads: blocks past the end read the last's.
PTA_HD int scale_block(int kb, int nk) { return kb < nk ? kb : nk - 1; }

} // namespace gemm_detail
} // namespace pta
