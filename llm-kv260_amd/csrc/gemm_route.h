// Which form an M > 1 product takes, from its sizes and the GPU's CU count.
// Free of HIP types so that a CPU test (tests/test_gemm_route.py) holds the
// rules against measured times.
#pragma once

namespace w4a8 {
namespace gemm_route {

// How many times the CUs are covered by the class-split kernel's items of 16
// rows x `tokens` tokens (gemm_mfma.hip). Its time goes in such steps: a CU's
// first item takes the latency of its rounds, each more about half of that.
inline long covers(int m, int rows, int cus, int tokens) {
    const long items = (long)((rows + 15) / 16) * ((m + tokens - 1) / tokens);
    return (items + cus - 1) / cus;
}

// Tokens per item of the class-split kernel, 16 or 32, for the same launch. A
// 32-token item takes 1.25 to 1.6 times a 16-token one's time.
//  * Two covers of 16 against one of 32: 32 (3072 x 2048 at 24 tokens 6.7
//    against 7.0 us, 3072 x 5888 17.1 against 21.6). But a round of a 16-token
//    item is four chunks where k allows it, of a 32-token one two, so 16 keeps
//    up on long rows: from k = 6144 it is up to 8% faster (2048 x 8192 at 33
//    tokens 15.4 against 16.3) where its rounds are even in number (they go in
//    pairs: at 7168 up to 6% slower). Past 64 tokens that starts at 8192 (900
//    x 6144 at 128: 14.8 against 13.6).
//  * As many covers of each, 16: 2560 x 8192 at 33 tokens 16.0 against 22.6.
//  * One cover more of 16: 16 with rounds of four chunks (3072 x 2048 at 64
//    tokens 8.3 against 9.4, 3072 x 8192 20.6 against 23.9), 32 where both
//    have the same rounds (k no multiple of 1024; 3333 x 3584 at 48 tokens
//    16.0 against 13.9). Two more, 32 (4096 x 8192 at 64 27.9 against 25.0).
inline int split_tokens(int m, int rows, int k, int cus) {
    const long n16 = covers(m, rows, cus, 16), n32 = covers(m, rows, cus, 32);
    if (m <= 16 || n16 <= 1) return 16;
    if (n32 == 1) return n16 == 2 && k >= (m > 64 ? 8192 : 6144) && k % 2048 == 0 ? 16 : 32;
    return n16 <= n32 + (k % 1024 == 0) ? 16 : 32;
}

// Rows per item of the class-split kernel for one token group, 16 or 8. Over
// long rows (k >= 8192: down), while 8-row items cover the CUs once: eight
// chunks a round, one workgroup a CU, 2048 x 8192 at 5 to 16 tokens in 9.2-10.1
// us against 10.4-10.6. Past that a CU runs two of them one after the other
// (3072 x 8192 at 16 16.2 against 10.5, 3072 x 16128 72 against 37), and at k =
// 2048 (o, q|k|v) they were slower too.
inline int split_rows(int m, int rows, int k, int cus) {
    return m <= 16 && k >= 8192 && (rows + 7) / 8 <= cus ? 8 : 16;
}

// Whether the whole-prompt kernel (gemm_tiles.hip) takes the product from the
// class-split kernel. One of its launches is one cover up to 64 tokens x 64
// rows a CU, at about 2.5 + 0.7 us a chunk: more than one or two of the
// class-split kernel's covers, less than three.
//  * Three covers of 32-token items and more: 2304 x 4096 at 160 tokens 15
//    against 18 us, 3072 x 5888 at 130 20 against 43.
//  * None of one cover (2048 x 8192 at 24 tokens 27 against 11), but for a
//    single chunk, where no round's latency hides another's: 64 x 256 at 6
//    tokens 3.1 against 3.4, 700 x 256 at 130 3.5 against 4.4; and past 64
//    tokens where rounds are one chunk, from about 45,000 outputs on: 300 x
//    1280 at 200 tokens 6.6 against 7.0, 16 x 2304 at 4,000 9.2 against 16.6
//    (64 x 2304 at 300 8.8 against 8.1).
//  * Two covers of 32, where rounds are one chunk (k no multiple of 512): 3333
//    x 2304 at 48 tokens 9.6 against 12.1. Else only on short rows, the
//    shorter the fewer 16-token items there are instead; up to 32 tokens on
//    shorter ones still, the weights then being most of its time (7168 x 3072
//    at 25 tokens 12.3 against 11.8, 3333 x 3072 at 72 11.7 against 15.4).
inline bool tiles_faster(int m, int rows, int k, int cus) {
    const long n16 = covers(m, rows, cus, 16), n32 = covers(m, rows, cus, 32);
    if (k == 256 || n32 >= 3) return true;
    if (n32 == 1) return k % 512 && m > 64 && (long)rows * m >= 45000;
    if (k % 512) return true;
    if (n16 == 2) return k < 1024;
    if (m <= 32) return k < 2048;
    return k < (n16 == 3 && k % 1024 == 0 ? 2048 : 4096);
}

enum Form { SPLIT, ROWS, TILES };   // gemm_mfma.hip, gemm_rows.hip, gemm_tiles.hip

// From ROWS_MIN rows on (and k a multiple of its 512-value segments) the
// row-split kernel takes up to 16 tokens: 8200 x 2048 7.1 us at 16 tokens
// against 9.3 in the whole-prompt kernel, which has 9.4 against 9.6 at 17;
// gate|up 8.1 and 9.9 at 16, 10.3 and 10.1 at 24; 32000 x 2048 13.6 and 14.4
// at 16, 18.6 and 14.4 at 17. (At 3,072 rows it was twice as slow as the
// class-split kernel: 48 workgroups.) Up to 32 tokens it stays ahead on longer rows while
// its workgroups of 64 rows are one cover of the CUs: 16384 x 8192 at 32
// tokens 28.5 against 31.6, 8192 x 16384 50.4 against 55.9; at k = 2048 even,
// and past one cover it loses (28672 x 8192 53.8 against 41.8).
constexpr int ROWS_MIN = 8192;

inline Form form(int m, int rows, int k, int cus) {
    if (rows >= ROWS_MIN && k % 512 == 0) {
        const bool two_tiles = m <= 32 && k >= 3072 && (rows + 63) / 64 <= cus;
        return m <= 16 || two_tiles ? ROWS : TILES;
    }
    return tiles_faster(m, rows, k, cus) ? TILES : SPLIT;
}

}  // namespace gemm_route
}  // namespace w4a8
