// Host-side walk over the buffer loads of the GEMM kernels (no device work).
#include "gemm_addr.h"

#include <algorithm>

#include "primus_turbo_amd.h"

namespace {
using namespace pta::gemm_detail;

// Whether n bytes at lane offset v and scalar offset s can be read past `end` (bytes
// from the descriptor's base) under one of the readings of the range check: the lane's
// offset alone, the sum, or the records less the scalar offset modulo 2^32.
bool stray(int32_t records, int32_t v, int32_t s, int n, int64_t end) {
    const uint64_t rec = static_cast<uint32_t>(records), lane = static_cast<uint32_t>(v), sum = lane + static_cast<uint32_t>(s);
    const bool     read = lane + n <= rec || sum + n <= rec ||
                      lane + n <= static_cast<uint32_t>(static_cast<uint32_t>(records) - static_cast<uint32_t>(s));
    return read && static_cast<int64_t>(sum) + n > end;
}

// operand [rows, K] of the 256 x 256 kernel; blocks past the last as the loops
// without the skip issue them
int64_t operand_strays(int64_t rows, int64_t K, int64_t ld, int tile) {
    const int nk = static_cast<int>((K + BK - 1) / BK);
    int64_t   n  = 0;
    for (int64_t r0 = 0; r0 < rows; r0 += tile)
        for (int h = 0; h < tile / HALF; ++h) {
            const int32_t rec = desc_records(half_bytes(half_rows(rows - r0, h), ld, K));
            const int64_t end = (rows - 1) * ld + K - (r0 + half_start(rows - r0, h)) * ld;
            for (int kb = 0; kb < nk + 2; ++kb)
                for (int r = 0; r < HALF; ++r)
                    for (int ch = 0; ch < BK / 16; ++ch) {
                        const bool oob = kb >= cut_block(nk, K) && past_k(nk, K, ch);
                        n += stray(item_records(rec, kb, nk), oob ? OOB_LANE : lane_off(r, ld, ch),
                                   item_soff(kb, nk), 16, end);
                    }
        }
    return n;
}

// scales of either kernel: es = 4 (fp32 per row and K block) or 1 (four E8M0 bytes)
int64_t scale_strays(int64_t rows, int64_t K, int es, bool two_d, int64_t sm, int64_t sk, int64_t bytes) {
    const int     nk = static_cast<int>((K + BK - 1) / BK);
    const int64_t up = (rows + BM - 1) / BM * BM;
    int64_t       n  = 0;
    for (int64_t r = 0; r < up; ++r)
        for (int kb = 0; kb < nk + 4; ++kb)
            n += stray(desc_records(bytes), scale_off(scale_row(r, rows), two_d, sm, es),
                       scale_block(kb, nk) * static_cast<int>(sk) * es, 4, bytes);
    return n;
}
} // namespace

extern "C" int64_t pta_test_gemm_stray_reads(int64_t rows, int64_t K, int64_t ld, int scale_elem_bytes, int scale_2d,
                                             int64_t s_m, int64_t s_k, int64_t s_bytes) {
    if (rows < 1 || K < 1 || ld < K) return -1;
    int64_t n = operand_strays(rows, K, ld, BM);
    if (scale_elem_bytes > 0) n += scale_strays(rows, K, scale_elem_bytes, scale_2d != 0, s_m, s_k, s_bytes);
    return n;
}
