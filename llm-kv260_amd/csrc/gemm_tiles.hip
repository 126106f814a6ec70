// Batched W4A8 for many tokens (a prompt): the results of gemm_mfma.hip and
// gemm_rows.hip, byte for byte (the contract's order, src/llm_kv260/q4_0.py:
// 170-182, applied row by row), a whole prompt in one launch.
//
// What bounds it: instruction issue. Every term of an output is a convert, two
// multiplies and an add in fp32, rounded in that order, against 32 MACs; the
// matrix cores need a third of the terms' time and the memory less. So:
//  * The convert and the first multiply are one fma. The MFMA adds its sums
//    16 sumi to the bits of MAGIC = 1.5 * 2^23, which then read as the float
//    F = MAGIC + 16 sumi (|16 sumi| <= 2^19, exact), and
//    fma(F, d_w / 16, -MAGIC * d_w / 16) is sumi * d_w rounded once: F and
//    the 13-bit product MAGIC * d_w / 16 are exact for every finite scale. An
//    infinite or NaN d_w gives NaN here, whatever the contract gives, in every
//    token of the row. So each wave looks at one token's accumulators before
//    the tree, and a workgroup with a NaN among them looks its rows' scales
//    over, and if one is not finite runs its tile once more by the contract's
//    own four operations: 2048 x 8192 at 512 tokens 40 us, 44 with every
//    output NaN from the activations, 79 with a bad scale in every row (each
//    NaN output by itself in one lane had taken 1,855). (A vote on the outputs
//    was 0.2 us a launch slower: a barrier of its own.)
//    With finite d_w the first product is the contract's, and so are NaNs from
//    d_x. Only a zero's sign may differ: an accumulator starts at +0.0f and
//    never sees it, and a NaN made of it and an infinite d_x has the same bits
//    either way.
//  * A wave's tile is 64 rows x 64 tokens (64 x 32 where that leaves CUs
//    idle), so that a block's weights are unpacked once for 64 tokens and
//    each operand read from LDS meets four MFMAs.
//  * A SIMD issues a VALU instruction every 2.6 clocks from two or more waves
//    in the VALU, one in 6.8 from a single one (measured), so it needs more
//    than two to choose from: two workgroups a CU, each running while the
//    other waits at its barrier or exchanges (one persistent workgroup of
//    eight waves, or of sixteen, with deeper prefetch: 41 and 43 us against
//    39 at 2048 x 8192 and 512 tokens, 155-157 against 131 at 2,048).
//  * 16x16x32 MFMAs: their results leave the VALU its rate, where a 32x32x32
//    one per 48 terms cost it a fifth. No DPP broadcasts of the scales: a DPP
//    multiply takes twice a plain one's time.
//
// A workgroup's eight waves share the tile, and wave w owns the contract's
// accumulator w: it takes the blocks 8c + w in increasing c and adds each
// term to its accumulator from +0.0f. At the end the eight accumulators of an
// output meet through LDS in the adjacent-pair tree.
//
// Operand layout of the 16x16x32 i8 MFMA (64 lanes):
//   A: lane l holds A[i = l % 16][k = 8 (l / 16) .. + 7]      (token i)
//   B: lane l holds B[k = 8 (l / 16) .. + 7][j = l % 16]      (row j)
//   D: lane l holds D[i = 4 (l / 16) + r][j = l % 16], r = 0..3
// The weight operand is 16 (n - 8) (gemm_rows.hip, block_weights).
//
// K goes by chunks of eight blocks, loaded straight into one of two LDS
// buffers while the other is computed: one barrier a chunk. The loads take no
// registers, which leaves the 128 of four waves a SIMD to the accumulators.
//
// Measured (MI355X, us; before: launches of 64 tokens through the kernels
// named above): gate|up (16384 x 2048) at 512 tokens 114 -> 69, at 2,048
// 451 -> 289; down (2048 x 8192) 127 -> 39 and 496 -> 131; q|k|v (3072 x 2048)
// 64 -> 21 and 255 -> 59; 3333 x 2304 at 333 tokens 107 -> 21.
#include "kernels.h"
#include "q4_0_device.h"

namespace w4a8 {

namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int WAVES = 8;                  // wave w owns accumulator w
constexpr int THREADS = 64 * WAVES;
constexpr int TILE_ROWS = 64;             // rows per workgroup
constexpr int RT = TILE_ROWS / 16;        // their MFMA tiles
constexpr uint32_t BUFFER_DWORD3 = 0x00020000;
constexpr int MAGIC_BITS = 0x4B400000;    // 1.5 * 2^23
constexpr float MAGIC = 12582912.0f;

struct TileParams {
    const uint8_t *w;
    const uint8_t *x;      // m rows, engine layout
    float *y;              // [m][rows]
    int rows;
    int k;
    int m;
    int x_stride;          // k + k / 8
    int per_xcd;           // items per XCD
    int items;
};

// An instance: NT token tiles of 16. LDS: RING chunk buffers, each the rows'
// 144 bytes, the tokens' 256 int8 and the tokens' 8 scales, as one stream of
// 1 KB pieces that the loads write; then the exchange of 32 tokens,
// [8 accumulators][64 rows][EXP tokens].
constexpr int RING = 2;
template <int NT>
struct TileGeo {
    static constexpr int TT = 16 * NT;
    static constexpr int WP = CHUNK_BYTES;       // sixteen rows' dwords fall on sixteen banks, four apart
    static constexpr int X_OFF = TILE_ROWS * WP;
    static constexpr int D_OFF = X_OFF + TT * 256;
    static constexpr int BUF = D_OFF + TT * 32;
    static constexpr int EXP = 32 + 4;
    static constexpr int EX_PART = TILE_ROWS * EXP * 4;
    static constexpr int LDS = RING * BUF > WAVES * EX_PART ? RING * BUF : WAVES * EX_PART;
    // A chunk's 1 KB loads: one of the weights' nine and X_LOADS of the
    // tokens' int8 in every wave, the weights' last in wave 0, the scales' in
    // the D_LOADS waves after it.
    static constexpr int X_LOADS = TT / 4 / WAVES;
    static constexpr int D_LOADS = TT / 32;
    static constexpr int LOADS = 1 + X_LOADS;    // of every wave; one more in the first 1 + D_LOADS
    static_assert(X_OFF == 1024 * (WAVES + 1) && TT % (4 * WAVES) == 0, "the loads below");
    static_assert(2 * (LDS + 1024) <= 160 * 1024, "two workgroups a CU, the flag and the vote's words among them");
};

template <int NT>
struct TileKernel {
    using G = TileGeo<NT>;

    // A lane's offset in each of its wave's loads.
    struct Slots {
        uint32_t w, x[G::X_LOADS], p;
        int p_lds;                        // the last load's offset in a buffer, -1 for none
    };
    static __device__ __forceinline__ void slots(const TileParams &P, int row_bytes, int w, int lane, Slots &s) {
        auto w_piece = [&](int q) {
            const int r = q / CHUNK_PIECES, p = q - CHUNK_PIECES * r;
            return (uint32_t)r * (uint32_t)row_bytes + 16u * (uint32_t)p;
        };
        s.w = w_piece(64 * w + lane);
#pragma unroll
        for (int i = 0; i < G::X_LOADS; ++i) {
            // Piece p of token t lies at 16-byte slot p ^ (t % 16), so that
            // sixteen tokens' reads of one piece fall on distinct banks.
            const int t = 4 * (G::X_LOADS * w + i) + (lane >> 4);
            s.x[i] = (uint32_t)t * (uint32_t)P.x_stride + 16u * (uint32_t)((lane ^ t) & 15);
        }
        // The scales of token 16 T + 4 g + e lie at 32-byte slot 16 T + 4 e + g:
        // a read takes the four tokens of one T and e, from distinct banks.
        const int slot = 32 * (w - 1) + (lane >> 1);
        const int t = (slot & ~15) + 4 * (slot & 3) + ((slot >> 2) & 3);
        s.p = w == 0 ? w_piece(64 * WAVES + lane) : (uint32_t)t * (uint32_t)P.x_stride + 16u * (uint32_t)(lane & 1);
        s.p_lds = w == 0 ? 1024 * WAVES : w <= G::D_LOADS ? G::D_OFF + 1024 * (w - 1) : -1;
    }

    // Where an item's chunks are loaded from. A row past the last or a token
    // past m lies beyond the resources' sizes and is not read (a lane's
    // offset says which row or token; the chunk's comes with the
    // instruction).
    struct Source {
        v4i w, x, p;
        int w_at, x_at, p_at, p_step;
    };
    static __device__ __forceinline__ v4i words(const uint8_t *base, uint32_t bytes) {
        const uint64_t b = (uint64_t)(uintptr_t)base;
        v4i r;
        r[0] = __builtin_amdgcn_readfirstlane((int)(uint32_t)b);
        r[1] = __builtin_amdgcn_readfirstlane((int)((uint32_t)(b >> 32) & 0xFFFFu));
        r[2] = __builtin_amdgcn_readfirstlane((int)bytes);
        r[3] = (int)BUFFER_DWORD3;
        return r;
    }
    static __device__ __forceinline__ void source(const TileParams &P, int row_bytes, int n0, int m0, int w, Source &S) {
        const uint32_t wn = (uint32_t)(P.rows - n0) * (uint32_t)row_bytes;
        const uint32_t xn = (uint32_t)(P.m - m0) * (uint32_t)P.x_stride;
        const uint8_t *wb = P.w + (size_t)n0 * row_bytes, *xb = P.x + (size_t)m0 * P.x_stride;
        S.w = words(wb, wn);
        S.x = words(xb, xn);
        S.p = words(w == 0 ? wb : xb + P.k, w == 0 ? wn : xn - (uint32_t)P.k);
        S.w_at = S.x_at = S.p_at = 0;
        S.p_step = w == 0 ? CHUNK_BYTES : 32;
    }

    // 1 KB straight into LDS: lane l's 16 bytes at `to` + 16 l. Written as
    // assembly because the compiler would wait for every load in flight before
    // the next LDS read; the waits are arrive()'s.
    static __device__ __forceinline__ void load_lds(const v4i &rsrc, uint32_t voff, int soff, int to) {
        // (the s_nop: m0 is written one wait state before a load reads it)
        __asm__ volatile("s_nop 0\n\tbuffer_load_dwordx4 %0, %1, %2 offen lds" ::"v"(voff), "s"(rsrc), "s"(soff), "{m0}"(to));
    }
    static __device__ __forceinline__ void load(const Slots &s, Source &S, int w, int buf) {
        load_lds(S.w, s.w, S.w_at, buf + 1024 * w);
#pragma unroll
        for (int i = 0; i < G::X_LOADS; ++i)
            load_lds(S.x, s.x[i], S.x_at, buf + G::X_OFF + 1024 * (G::X_LOADS * w + i));
        if (s.p_lds >= 0) load_lds(S.p, s.p, S.p_at, buf + s.p_lds);
        S.w_at += CHUNK_BYTES;
        S.x_at += 256;
        S.p_at += S.p_step;
    }
    // Every wave's loads have landed.
    static __device__ __forceinline__ void arrive() {
        __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
    }

    // Per-lane offsets of the operands of block b of a chunk. The lane takes
    // weights 8 g .. 8 g + 7 (g = lane / 16): the low (g < 2) or high nibbles
    // of bytes 8 (g % 2) .. + 7 of the block's run. An even block starts at a
    // dword boundary, its nibbles two bytes in; an odd block two bytes into a
    // dword, its nibbles in the next. Dword e of the operand is 32 bits of the
    // dwords at `nib` from bit 32 e + shift on, so that the wanted nibble of
    // each byte lies in its high half: for the low nibbles from four bits
    // before the block's run, for the high ones from the run.
    struct Lane {
        int nib, scl, xa, dx;
        uint32_t shift;
    };
    static __device__ __forceinline__ Lane lane_offsets(int b, int lane) {
        const int j = lane & 15, g = lane >> 4, up = g >> 1, odd = b & 1;
        Lane L;
        L.scl = j * G::WP + 18 * b;
        L.nib = L.scl + 8 * (g & 1) + (odd ? (up ? 2 : -2) : 0);
        L.shift = odd ? (up ? 0u : 28u) : (up ? 16u : 12u);
        L.xa = G::X_OFF + 256 * j + 16 * ((2 * b + up) ^ j) + 8 * (g & 1);
        L.dx = G::D_OFF + 32 * g + 4 * b;
        return L;
    }

    // One block's terms, added to the wave's accumulator; PLAIN by the
    // contract's operations as written. `bias` is what the MFMAs add their
    // sums to: MAGIC's bits, or 0 if PLAIN.
    template <bool PLAIN>
    static __device__ __forceinline__ void block(const uint8_t *buf, const Lane &L, const v4i &bias, float acc[NT][RT][4]) {
        long wb[RT];
        float dw[RT], dm[RT];
#pragma unroll
        for (int r = 0; r < RT; ++r) {
            const uint32_t *n = reinterpret_cast<const uint32_t *>(buf + L.nib + 16 * r * G::WP);
            const uint32_t half = *reinterpret_cast<const uint16_t *>(buf + L.scl + 16 * r * G::WP);
            const uint32_t v0 = n[0], v1 = n[1], v2 = n[2];
            const uint32_t lo = (__builtin_amdgcn_alignbit(v1, v0, L.shift) & 0xF0F0F0F0u) ^ 0x80808080u;
            const uint32_t hi = (__builtin_amdgcn_alignbit(v2, v1, L.shift) & 0xF0F0F0F0u) ^ 0x80808080u;
            wb[r] = (long)(((uint64_t)hi << 32) | lo);
            dw[r] = half_bits_to_float(half) * 0.0625f;
            dm[r] = dw[r] * -MAGIC;
        }
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const long ax = *reinterpret_cast<const long *>(buf + L.xa + 16 * t * 256);
            float dx[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) dx[e] = *reinterpret_cast<const float *>(buf + L.dx + (16 * t + 4 * e) * 32);
            v4i d[RT];
#pragma unroll
            for (int r = 0; r < RT; ++r) d[r] = __builtin_amdgcn_mfma_i32_16x16x32_i8(ax, wb[r], bias, 0, 0, 0);
#pragma unroll
            for (int r = 0; r < RT; ++r)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float a = PLAIN ? (float)d[r][e] * dw[r] : __builtin_fmaf(__int_as_float(d[r][e]), dw[r], dm[r]);
                    acc[t][r][e] = acc[t][r][e] + a * dx[e];
                }
        }
    }

    // Exchange of token tiles 2 h and 2 h + 1: the tree over the eight
    // accumulators, and the stores.
    static __device__ __forceinline__ void reduce_half(const TileParams &P, int n0, int m0, uint8_t *ex, int w, int lane, int h,
                                                       const float acc[NT][RT][4]) {
        const int j = lane & 15, g = lane >> 4;
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int r = 0; r < RT; ++r)
                *reinterpret_cast<float4 *>(ex + w * G::EX_PART + ((16 * r + j) * G::EXP + 16 * t + 4 * g) * 4) =
                    make_float4(acc[2 * h + t][r][0], acc[2 * h + t][r][1], acc[2 * h + t][r][2], acc[2 * h + t][r][3]);
        __syncthreads();
        // Wave w takes tokens 4 w .. 4 w + 3, a row a lane.
        const int row = n0 + lane, tok = m0 + 32 * h + 4 * w;
        float4 l[8];
#pragma unroll
        for (int b = 0; b < 8; ++b)
            l[b] = *reinterpret_cast<const float4 *>(ex + b * G::EX_PART + (lane * G::EXP + 4 * w) * 4);
        const float v[4] = {((l[0].x + l[1].x) + (l[2].x + l[3].x)) + ((l[4].x + l[5].x) + (l[6].x + l[7].x)),
                            ((l[0].y + l[1].y) + (l[2].y + l[3].y)) + ((l[4].y + l[5].y) + (l[6].y + l[7].y)),
                            ((l[0].z + l[1].z) + (l[2].z + l[3].z)) + ((l[4].z + l[5].z) + (l[6].z + l[7].z)),
                            ((l[0].w + l[1].w) + (l[2].w + l[3].w)) + ((l[4].w + l[5].w) + (l[6].w + l[7].w))};
        if (row < P.rows) {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (tok + e < P.m) P.y[(size_t)(tok + e) * P.rows + row] = v[e];
        }
    }

    // The item at rows n0 .., tokens m0 ..: chunk c is computed from LDS
    // buffer c % 2 while the loads of chunk c + 1 fill the other. Sets *nan
    // (0 before) if a row's first token is NaN in a wave's accumulator.
    template <bool PLAIN>
    static __device__ __forceinline__ void pass(const TileParams &P, int n0, int m0, uint8_t *lds, int *nan) {
        const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
        int lane = threadIdx.x & 63;
        if constexpr (PLAIN) __asm__ volatile("" : "+v"(lane));   // else the first pass's offsets are kept for this one, and spill
        const int row_bytes = P.k / QK * Q4_0_BYTES;
        const int chunks = P.k / 256;
        const int base = (int)(uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)lds;
        Slots s;
        slots(P, row_bytes, w, lane, s);
        Source S;
        source(P, row_bytes, n0, m0, w, S);
        load(s, S, w, base);
        const Lane L = lane_offsets(w, lane);
        constexpr int BIAS = PLAIN ? 0 : MAGIC_BITS;
        v4i bias = {BIAS, BIAS, BIAS, BIAS};
        __asm__ volatile("" : "+v"(bias));
        float acc[NT][RT][4];
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int r = 0; r < RT; ++r)
#pragma unroll
                for (int v = 0; v < 4; ++v) acc[t][r][v] = 0.0f;
        arrive();
        for (int c = 0;; c += RING) {
            if (c + 1 < chunks) load(s, S, w, base + G::BUF);   // last read for chunk c - 1, before the last barrier
            block<PLAIN>(lds, L, bias, acc);
            arrive();
            if (c + 1 >= chunks) break;
            if (c + 2 < chunks) load(s, S, w, base);
            block<PLAIN>(lds + G::BUF, L, bias, acc);
            arrive();
            if (c + 2 >= chunks) break;
        }
        if constexpr (!PLAIN) {
            bool any = false;
#pragma unroll
            for (int r = 0; r < RT; ++r) any = any || acc[0][r][0] != acc[0][r][0];
            if (any) *nan = 1;
        }
#pragma unroll
        for (int h = 0; h < NT / 2; ++h) {
            if (h) __syncthreads();                              // the half before is read
            reduce_half(P, n0, m0, lds, w, lane, h, acc);
        }
    }

    // Whether one of the blocks this thread looks at (a row's b, b + 8, ..) has a scale that is not finite.
    static __device__ __forceinline__ bool scale_not_finite(const TileParams &P, int n0) {
        const int row = n0 + ((int)threadIdx.x >> 3), nb = P.k / QK;
        if (row >= P.rows) return false;
        const uint8_t *src = P.w + (size_t)row * ((size_t)nb * Q4_0_BYTES);
        bool bad = false;
#pragma unroll 8
        for (int b = threadIdx.x & 7; b < nb; b += 8)
            bad |= (*reinterpret_cast<const uint16_t *>(src + (size_t)b * Q4_0_BYTES) & 0x7C00u) == 0x7C00u;
        return bad;
    }

    static __device__ __forceinline__ void run(const TileParams &P, int n0, int m0, uint8_t *lds, int *nan) {
        if (threadIdx.x == 0) *nan = 0;                          // before the barriers of the chunks
        pass<false>(P, n0, m0, lds, nan);
        if (*nan == 0) return;                                   // set before the exchange's barrier
        // (the vote's barriers keep the exchange until every wave has read it)
        if (__syncthreads_or(scale_not_finite(P, n0))) pass<true>(P, n0, m0, lds, nan);
    }
};
static_assert(THREADS == 8 * TILE_ROWS, "scale_not_finite: eight threads a row");

template <int NT>
__global__ __launch_bounds__(THREADS) __attribute__((amdgpu_waves_per_eu(4, 4))) void gemm_tiles_kernel(TileParams P) {
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    __shared__ int nan;
    // Workgroups go to the XCDs in turn: each XCD takes a contiguous run of
    // items, token groups fastest, so its L2 serves a row group's weights to
    // all token groups and the activations to all its row groups.
    const int item = (int)(blockIdx.x & 7) * P.per_xcd + (int)(blockIdx.x >> 3);
    if (item >= P.items) return;
    const int tgs = (P.m + 16 * NT - 1) / (16 * NT);
    const int rg = item / tgs;
    const int n0 = rg * TILE_ROWS, m0 = (item - rg * tgs) * 16 * NT;
    // A last group of at most 32 tokens works on 32.
    if (NT == 4 && P.m - m0 <= 32)
        TileKernel<2>::run(P, n0, m0, lds, &nan);
    else
        TileKernel<NT>::run(P, n0, m0, lds, &nan);
}

template <int NT>
hipError_t launch_tiles(TileParams P, hipStream_t stream) {
    using G = TileGeo<NT>;
    const auto kernel = &gemm_tiles_kernel<NT>;
    const hipError_t e = allow_dynamic_lds(reinterpret_cast<const void *>(kernel), 160 * 1024);
    if (e != hipSuccess) return e;
    const long items = (long)((P.rows + TILE_ROWS - 1) / TILE_ROWS) * ((P.m + G::TT - 1) / G::TT);
    if (items > 0x0fffffffL) return hipErrorInvalidValue;
    P.items = (int)items;
    P.per_xcd = (int)((items + 7) / 8);
    hipLaunchKernelGGL(kernel, dim3((unsigned)(8 * P.per_xcd)), dim3(THREADS), G::LDS, stream, P);
    return hipGetLastError();
}

}  // namespace

hipError_t launch_gemm_tiles(const uint8_t *w, const uint8_t *x, int m, float *y, int rows, int k, int cus,
                             hipStream_t stream) {
    TileParams P{};
    P.w = w;
    P.x = x;
    P.y = y;
    P.rows = rows;
    P.k = k;
    P.m = m;
    P.x_stride = k + k / 8;
    // 32-token tiles while every CU gets at most one: a lone workgroup's time
    // is its chunks' (2048 x 8192 at 256 tokens: 26 us against 37). Past that
    // 64-token tiles, 4% slower to 25% faster (gate|up 8% at 512 tokens).
    const long row_groups = (rows + TILE_ROWS - 1) / TILE_ROWS;
    if (row_groups * ((m + 31) / 32) <= cus) return launch_tiles<2>(P, stream);
    return launch_tiles<4>(P, stream);
}

}  // namespace w4a8
