// bamd_dense.hip — products with dense bfloat16 matrices in the packed layout of bamd_dense.h.
//   dense_tile_kernel: many rows (prompts).  Weight and activation tiles global -> LDS by DMA, four or eight stages deep, under the matrix instructions.
//   dense_few_kernel: up to 64 rows (decoding several sequences, short prompts), bfloat16; its rows may lie by blocks.  The waves of a block split K, each with a DMA ring of weights and rows.
//   dense_mv_kernel: a row (decoding), and up to 64 in three parts (32-bit).  The eight or sixteen waves of a block split K; every wave streams its share of a 16-row tile straight from HBM into matrix operands.  With
//     a single row the mechanism in front of the product (residual + norm + token shift or layer norms, PolyNorm, clamped gated unit, grouped norm, last norm) runs as its prologue, its weights
//     already requested.
#include "bamd_dense_device.h"
#include "bamd_mfma_common.h"
#include <algorithm>
#include <limits.h>
#include <type_traits>

// ---- packing at load: value (row, col) of the packed matrix = src[row_off[row] + col_off[col]], zero where either is negative; row tiles go to every step-th row tile of
// a matrix of ld column blocks ------------------------------------------------------------------------------------------------------------------------------
__global__ void __launch_bounds__(64) pack_kernel(const uint16_t * src, const int32_t * row_off, const int32_t * col_off, int k_tiles, uint16_t * dst, int step, int ld) {
    const int lane = threadIdx.x, kt = blockIdx.x % k_tiles, rt = blockIdx.x / k_tiles;
    const int ro = row_off[rt * 16 + (lane & 15)];
    uint16_t * d = dst + (((size_t) rt * step * ld + kt) * 64 + lane) * 8;
    for (int i = 0; i < 8; ++i) { const int co = col_off[kt * 32 + (lane >> 4) * 8 + i]; d[i] = ro < 0 || co < 0 ? 0 : src[(size_t) ro + co]; }
}
void bamd_launch_pack(const uint16_t * src, const int32_t * row_off, const int32_t * col_off, int row_tiles, int k_tiles, uint16_t * dst, int step, int ld, hipStream_t s) {
    hipLaunchKernelGGL(pack_kernel, dim3(row_tiles * k_tiles), dim3(64), 0, s, src, row_off, col_off, k_tiles, dst, step, ld);
}

// ---- many rows --------------------------------------------------------------------------------------------------------------------------------------
// one 16 x 16 result tile of a wave: activation rows from mb, matrix rows from nb; a: the tiles of the same activation rows, j: which one
template <typename T, int OUT, int NI>
__device__ __forceinline__ void store_tile(const bamd_v4 (&a)[NI], int j, int mb, int nb, int n_lim, int n_rows, int rows, void * out, int ldo, int cbo, float limit, int lane) {
    if (nb >= n_lim) return;
    if constexpr (OUT == BAMD_OUT_ACT_T) {
        const int n = nb + (lane & 15), m = mb + (lane >> 4) * 4;
        if (n >= n_rows) return;
#pragma unroll
        for (int k = 0; k < 4; ++k) if (m + k < rows) ((T *) out)[(size_t) n * ldo + m + k] = to_act<T>(a[j][k]);
    } else if constexpr (OUT == BAMD_OUT_GLU) {                   // tiles in turn: gate, up
        const int n = (nb >> 1) + (lane >> 4) * 4, m = mb + (lane & 15);
        if ((j & 1) || m >= rows) return;
        bamd_v4 o;
#pragma unroll
        for (int k = 0; k < 4; ++k) o[k] = clamped_glu(a[j][k], a[j | 1][k], limit);
        store4<Operand<T>>(row_out<Operand<T>>(out, m, ldo, cbo).at(n), o);
    } else {
        const int n = nb + (lane >> 4) * 4, m = mb + (lane & 15);
        if (m >= rows) return;
        if constexpr (OUT == BAMD_OUT_F32) {
            float * o = (float *) out + (size_t) m * ldo + n;
            if (n + 3 < n_rows) *(bamd_v4 *) o = a[j];
            else for (int k = 0; k < 4; ++k) if (n + k < n_rows) o[k] = a[j][k];
        } else {
            T * o = (T *) out + (size_t) m * ldo + n;
#pragma unroll
            for (int k = 0; k < 4; ++k) if (n + k < n_rows) o[k] = to_act<T>(a[j][k]);
        }
    }
}
// 32-bit: weights are bfloat16, activations three planes of it (bamd_dense_device.h), and products of bfloat16 numbers are exact in 32 bits: three bfloat16 matrix instructions do what eight of
// 16x16x4_f32 did, with three roundings of a sum per 32 columns for thirty-two.
// rows [rows][ldx] of 32 k_tiles floats -> operand rows by blocks (rows that no kernel writes as operands: cached latents, of which a pass may have more than a grid's y axis takes)
__global__ void __launch_bounds__(256) split_rows_kernel(const float * __restrict__ x, int ldx, int k_tiles, void * planes, int cb) {
    const int i = (blockIdx.y * 256 + threadIdx.x) * 4;
    if (i < k_tiles * 32) store4<bamd_s3>(row_out<bamd_s3>(planes, blockIdx.x, 0, cb).at(i), *(const bamd_v4 *) (x + (size_t) blockIdx.x * ldx + i));
}
void bamd_launch_split_rows(const float * x, int ldx, int rows, int k_tiles, void * planes, int cb, hipStream_t s) {
    hipLaunchKernelGGL(split_rows_kernel, dim3(rows, (k_tiles * 8 + 255) / 256), dim3(256), 0, s, x, ldx, k_tiles, planes, cb);
}
// TM activation rows x TN matrix rows per block of WM x WN waves.  Both operands travel global -> LDS by DMA (a kilobyte per instruction: 16 rows x 32 columns), NS stages
// of 32 columns deep: while the matrix instructions of column block k run from registers, the fragments of k + 1 are read from LDS and the copies of the NS - 2 blocks
// behind it are under way; one barrier per column block, which waits for copies issued NS - 2 blocks ago.  What bounded the kernel before it (128 x 128, staged through registers) was LDS
// traffic: a wave tile of 64 x 64 reads as many bytes per matrix instruction as 128 x 64 does per 1.3.  Reads and copies are spread between the rows of matrix instructions:
// all of them in front of the first costs 15 %.
// Activations lie in LDS as they come from memory, four lanes on 64 consecutive bytes of a row (one 16-byte piece of 16 rows per four lanes costs the vector memory path
// four times the lookups: 446 -> 409 us below), the pieces of a row turned by half its number: sixteen rows of one piece then fall on different banks.
// Rows by blocks (bamd_dense.h), 2048 of them: 256 x 256 tiles 0 to 4 % (8448 outputs 319 -> 305 us), 128 x 256 6 to 7 % (149 -> 138).
// 32-bit (three planes of activations): the sums of a column block start at zero and are added to the accumulators by the vector units, a row of tiles behind.  The matrix instructions cut off
// where the vector units round: kept in them from one column block to the next, a sum of 14336 positive products was off by 6.3e-6 (1.8e-6 with the f32 instructions), so it is 3.2e-7 (and
// 4.1e-7 for 2.2e-6 with random signs).  500 x 8192 x 2048 118 -> 46 us, 500 x 12608 x 2048 178 -> 75, 500 x 2048 x 8192 122 -> 63.
// 2048 x 28672 x 4096: 676 -> 409 us (1176 TFLOP/s); 2048 x 4096 x 14336: 284 -> 185 us (1303); 2048 x 2048 x 2048: 41 -> 22 us; 131 x 8192 x 2048: 23 -> 16 us.
__device__ __forceinline__ const unsigned char * uniform_at(const unsigned char * p) {
    return (const unsigned char *) ((uint64_t) (uint32_t) __builtin_amdgcn_readfirstlane((int) (uint32_t) (uint64_t) p) | (uint64_t) (uint32_t) __builtin_amdgcn_readfirstlane((int) ((uint64_t) p >> 32)) << 32);
}
template <typename T, int TM, int TN, int WM, int WN, int NS, int OUT>
__global__ void __launch_bounds__(64 * WM * WN) dense_tile_kernel(bamd_dense w, const bamd_bf * x, int ldx, int cb, int rows, void * out, int ldo, int cbo, int n_mt, int n_nt, float limit) {
    const int kb = (int) ((long) w.k_tiles * blockIdx.y / gridDim.y), nk = (int) ((long) w.k_tiles * (blockIdx.y + 1) / gridDim.y) - kb;      // this block's share of K
    constexpr int XT = TM / 16, WT = TN / 16, NW = WM * WN, MI = XT / WM, NI = WT / WN, XP = bamd_planes<T>, UNITS = XT * XP + WT, PER = (UNITS + NW - 1) / NW, STAGE = UNITS * 1024;
    static_assert((XP == 1 || MI % 2 == 0) && MI * WM == XT && NI * WN == WT && NS >= 4 && (NS & (NS - 1)) == 0 && (OUT != BAMD_OUT_GLU || NI % 2 == 0), "");
    extern __shared__ __align__(16) unsigned char lds[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int total = n_mt * n_nt;
    int id = blockIdx.x;
    { const int per = (total + 7) / 8, xcd = id & 7, k = id >> 3; id = xcd * per + k; if (k >= per || id >= total) return; }
    const int mt = id % n_mt, nt = id / n_mt, m0 = mt * TM, n0t = nt * WT;
    // this wave's share of a stage: PER of its kilobytes, of activations and then of weights (past the last one: that one again)
    const unsigned char * src[PER]; uint32_t off[PER], step[PER], dst[PER];
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int u = i * NW + wave < UNITS ? i * NW + wave : UNITS - 1;
        dst[i] = (uint32_t) (size_t) (bamd_lds_vp) lds + (uint32_t) u * 1024u;
        if (u < XT * XP) {                                        // 16 rows of four 16-byte pieces, of one plane
            int row = u / XP * 16 + (lane >> 2);
            row = m0 + row < rows ? row : rows - 1 - m0;
            src[i] = uniform_at((const unsigned char *) (x + (size_t) m0 * ldx + (size_t) kb * cb)); step[i] = (uint32_t) cb * 2u;
            off[i] = (uint32_t) row * (uint32_t) ldx * 2u + (uint32_t) (u % XP) * 64u + (uint32_t) ((lane & 3) ^ ((lane >> 3) & 3)) * 16u;
        } else {
            int tile = u - XT * XP;
            tile = n0t + tile < w.row_tiles ? tile : w.row_tiles - 1 - n0t;
            src[i] = uniform_at((const unsigned char *) (w.w + ((size_t) n0t * w.k_tiles + kb) * 512)); step[i] = 1024u;
            off[i] = (uint32_t) tile * (uint32_t) w.k_tiles * 1024u + (uint32_t) lane * 16u;
        }
    }
    // copy i of PER of stage k (behind the last column block: the last one again, into a stage nobody reads)
    auto copy = [&](int k, int i) {
        const int kk = k < nk ? k : nk - 1;
        lds_dma16_s(src[i] + (size_t) kk * step[i], off[i], dst[i] + (uint32_t) (k & (NS - 1)) * STAGE);
    };
    const int wm = wave % WM, wn = wave / WM;
    const int r = lane & 15, q = lane >> 4;                       // the lane's row of a block and its eight columns
    const unsigned char * xb = lds + (size_t) wm * MI * XP * 1024 + (r * 4 + (q ^ ((r >> 1) & 3))) * 16, * wb = lds + (size_t) (XT * XP + wn * NI) * 1024 + lane * 16;
    bamd_v4 acc[MI][NI];
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NI; ++j) acc[i][j] = bamd_v4{ 0, 0, 0, 0 };
    bamd_v4 part[2][NI];                                          // 32-bit: the sums of a column block, of this row of tiles and the one in front
#pragma unroll
    for (int j = 0; j < NI; ++j) part[(MI - 1) & 1][j] = bamd_v4{ 0, 0, 0, 0 };
    auto add = [&](int i) {
#pragma unroll
        for (int j = 0; j < NI; ++j) acc[i][j] = acc[i][j] + part[i & 1][j];
    };
    bamd_bf8 xf[2][MI][XP], wf[2][NI];
    auto read_x = [&](int k, int p, int i, int c) { xf[p][i][c] = *(const bamd_bf8 *) (xb + (k & (NS - 1)) * STAGE + (i * XP + c) * 1024); };
    auto read_w = [&](int k, int p, int j) { wf[p][j] = *(const bamd_bf8 *) (wb + (k & (NS - 1)) * STAGE + j * 1024); };
    auto wait = [&] {                                             // in block k: leaves NS - 3 stages of this wave's copies under way, so that stage k + 1 is whole; then every wave's
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" :: "n"((NS - 3) * PER) : "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    auto block = [&](int k, auto par) {
        constexpr int P = decltype(par)::value;
        wait();                                                   // stage k + 1 is whole; stage k - 1 is free
        // MI groups: a row of matrix instructions, and spread over them the copies of stage k + NS - 1 and the reads of stage k + 1
#pragma unroll
        for (int i = 0; i < MI; ++i) {
#pragma unroll
            for (int c = i * PER / MI; c < (i + 1) * PER / MI; ++c) copy(k + NS - 1, c);
#pragma unroll
            for (int j = i * NI / MI; j < (i + 1) * NI / MI; ++j) read_w(k + 1, P ^ 1, j);
#pragma unroll
            for (int c = 0; c < XP; ++c) read_x(k + 1, P ^ 1, i, c);
#pragma unroll
            for (int c = XP - 1; c >= 0; --c)                     // the smallest parts first
#pragma unroll
                for (int j = 0; j < NI; ++j) {
                    const bamd_v4 from = XP == 1 ? acc[i][j] : c == XP - 1 ? bamd_v4{ 0, 0, 0, 0 } : part[i & 1][j];
                    bamd_v4 & to = XP == 1 ? acc[i][j] : part[i & 1][j];
                    if constexpr (OUT == BAMD_OUT_ACT_T) to = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xf[P][i][c], wf[P][j], from, 0, 0, 0);      // lane: four activation rows of one matrix row
                    else to = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[P][j], xf[P][i][c], from, 0, 0, 0);                                       // lane: four matrix rows of one activation row
                }
            if constexpr (XP > 1) add(i ? i - 1 : MI - 1);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
#pragma unroll
    for (int st = 0; st < NS - 1; ++st)
#pragma unroll
        for (int i = 0; i < PER; ++i) copy(st, i);
    asm volatile("s_waitcnt vmcnt(%0)" :: "n"((NS - 2) * PER) : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int c = 0; c < XP; ++c) read_x(0, 0, i, c);
#pragma unroll
    for (int j = 0; j < NI; ++j) read_w(0, 0, j);
    int k = 0;
    for (; k + 2 <= nk; k += 2) { block(k, std::integral_constant<int, 0>()); block(k + 1, std::integral_constant<int, 1>()); }
    if (k < nk) block(k, std::integral_constant<int, 0>());
    if constexpr (XP > 1) add(MI - 1);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");              // (no copy outlives the block)
    const int n_lim = w.row_tiles * 16;
    if constexpr (OUT == BAMD_OUT_F32) out = (float *) out + (size_t) blockIdx.y * rows * ldo;
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NI; ++j) store_tile<T, OUT>(acc[i], j, m0 + (wm * MI + i) * 16, (n0t + wn * NI + j) * 16, n_lim, w.rows, rows, out, ldo, cbo, limit, lane);
}
template <typename T, int TM, int TN, int WM, int WN, int NS, int OUT>
static int tile_go(const bamd_dense & w, const void * x, int ldx, int cb, int rows, void * out, int ldo, int cbo, float limit, int parts, hipStream_t s) {
    const int n_mt = (rows + TM - 1) / TM, n_nt = (w.row_tiles + TN / 16 - 1) / (TN / 16), per = (n_mt * n_nt + 7) / 8;
    hipLaunchKernelGGL((dense_tile_kernel<T, TM, TN, WM, WN, NS, OUT>), dim3(per * 8, parts), dim3(64 * WM * WN), (size_t) NS * (TM / 16 * bamd_planes<T> + TN / 16) * 1024, s, w, (const bamd_bf *) x, ldx, cb, rows, out, ldo, cbo, n_mt, n_nt, limit);
    return 0;
}
// The tile whose rounds over the 256 CUs end first.  Measured per block of 32 columns (ns), half of the CUs busy and all: 256 x 256 650 to 785, 256 x 224 630 to 740, 256 x 192 565 to 655, 256 x 160
// 512 to 572, 128 x 256 432 to 490, 128 x 128 250 (280 in several rounds), all of them one block per CU, so that a round started is a round paid: the widths between are there for what 256 leaves over.  2048 x 16896 x
// 4096 (66 tiles of 256 in two rows of rounds and a bit) 289 -> 258 us on 192, 2048 x 4736 x 4096 94 -> 74 on 160, 1485 x 14336 x 4096 192 -> 164 on 192, 2048 x 14336 x 4096 206 -> 198 on 224; over 23
// sizes the choice is 0.3 % behind the best on average (7 % without them); of 53 others where they change it, it is 16 % ahead on average and 3 % behind at worst.  64 x 128 195 and 64 x 64 160 share a CU with two to four others and never take less than 250 and 160.  Where even the small tiles leave
// CUs idle and the reader of the result can add planes, K is halved: two planes cost their bytes twice (at 4 TB/s) and blocks their
// start and end once more (4 us).  131 x 2048 x 8192: 38 -> 22 us, 412 x 4096 x 8192: 85 -> 39; four shares were no faster (24 and 43 us).  Halves of 64 x 64 tiles that put a second block on
// a CU take 300 where each half is longer than 2048 columns: 131 x 4096 x 14336 whole 70 us, in halves of such tiles 74, of 128 x 128 58 (8192 columns: 41, 43, 36); at K = 4096 they are
// level or ahead (131 x 3072: 24.0 and 24.4, 300 x 2048: 24.4 and 19.9).  Of 187 halved sizes (K 1056 to 14336) nine are slower than whole by more than 2 %, at most 7 % (17 and 11 % without).
// 32-bit, three planes of activations: a block of 128 x 256 takes 800 ns where few CUs are busy and 1280 where all are (their copies out of L2), 128 x 128 430 and 690, 64 x 128 370 and 460, two of them
// on a CU 700 to 800, 64 x 64 250 and 300, four on a CU 1000.  Halves: only what the reader of the second plane pays.  Of 94 choices (512 to 12608 outputs, K 512 to 14336, 70 to 2048 rows) the mean is
// 0.5 % behind the best and the worst 10 %
enum { TILE_256_256 = 0, TILE_128_256 = 1, TILE_128_128 = 2, TILE_64_128 = 3, TILE_64_64 = 4, TILE_64_64_DEEP = 5, TILE_256_224 = 6, TILE_256_192 = 7, TILE_256_160 = 8 };
static int pick_tile(int act, const bamd_dense & w, int rows, int most, int & share, int out, long * cost = nullptr) {
    share = 1;
    auto tiles = [&](int tm, int tn) { return (long) ((rows + tm - 1) / tm) * ((w.row_tiles * 16 + tn - 1) / tn); };
    long best = 0; int pick = 0;
    if (act == BAMD_ACT_F32) {
        static const int kind[4] = { TILE_128_256, TILE_128_128, TILE_64_128, TILE_64_64 };
        for (int p = 1; p <= most && p <= 2 && (p == 1 || w.k_tiles >= 32); ++p) {
            auto rounds = [](long b, long lo, long by) { return b / 256 * (lo + by) + (b % 256 ? lo + by * (b % 256) / 256 : 0); };
            const long b1 = tiles(64, 128) * p, b0 = tiles(64, 64) * p;
            const long t[4] = { rounds(tiles(128, 256) * p, 800, 480), rounds(tiles(128, 128) * p, 430, 260), std::max(b1 > 256 ? 700 : 370 + 90 * b1 / 256, 400 * b1 / 256), std::max(250 + 50 * b0 / 256, 250 * b0 / 256) };
            const int i = (int) (std::min_element(t, t + 4) - t);
            const long ns = t[i] * ((w.k_tiles + p - 1) / p) + (p > 1 ? (long) rows * w.row_tiles * 16 / 1000 : 0);
            if (p == 1 || ns < best) { best = ns; pick = kind[i]; share = p; }
        }
        return pick;
    }
    for (int p = 1; p <= most && p <= 2 && (p == 1 || w.k_tiles >= 32); ++p) {
        auto rounds = [&](int tm, int tn, long lo, long by) { const long b = tiles(tm, tn) * p; return b / 256 * (lo + by) + (b % 256 ? lo + by * std::max(0l, b % 256 - 128) / 128 : 0); };
        const long pairs = p == 2 && w.k_tiles > 128 && tiles(64, 64) * 2 > 256 ? 300 : 160;
        const bool odd = p == 1 && out != BAMD_OUT_GLU;           // gate and up tiles lie in turn: a wave holds an even number
        const long t[8] = { rounds(256, 256, 650, 135), rounds(128, 256, 432, 58), tiles(128, 128) * p <= 256 ? 250 : rounds(128, 128, 250, 30), std::max(tiles(64, 128) * p * 195 / 256, 250l), std::max(tiles(64, 64) * p * 160 / 256, pairs),
                            odd ? rounds(256, 224, 630, 110) : LONG_MAX, p == 1 ? rounds(256, 192, 565, 90) : LONG_MAX, odd ? rounds(256, 160, 512, 60) : LONG_MAX };
        static const int kind[8] = { TILE_256_256, TILE_128_256, TILE_128_128, TILE_64_128, TILE_64_64, TILE_256_224, TILE_256_192, TILE_256_160 };
        const int i = (int) (std::min_element(t, t + 8) - t);
        const long ns = t[i] * ((w.k_tiles + p - 1) / p) + (p > 1 ? 4000 + (long) p * rows * w.row_tiles * 16 / 500 : 0);
        if (p == 1 || ns < best) { best = ns; pick = kind[i]; share = p; }
    }
    if (cost) *cost = best;
    // one tile per CU at most: twice the stages hide more of the memory's latency (131 x 2048 x 8192: 49 -> 38 us); with more, blocks hide each other's
    return pick == TILE_64_64 && tiles(64, 64) * share <= 256 ? TILE_64_64_DEEP : pick;
}
// Row tiles of the matrix that whole rounds of 256 x 256 take, the rest going to a product of its own, where that is ahead by more than 3 % (of one product; halves are not cut): 0 none.  The launch
// between them is 4 us.  2048 x 28672 x 4096 with the gated unit (3.5 rounds) 377 -> 352 us; 2048 x 16896 x 4096 249 -> 239.  Only for numbers of row tiles that divide the CUs: a round of others leaves
// some idle, and what a cut gives there has not been measured
int bamd_dense_cut(const bamd_dense & w, int rows, int out) {
    const int n_mt = (rows + 255) / 256;
    if (256 % n_mt) return 0;
    const int per = 256 / n_mt * 16, full = w.row_tiles / per * per;      // row tiles of a round
    if (!full || full == w.row_tiles) return 0;
    bamd_dense a = w, b = w; int share; long whole, ca, cb;
    a.row_tiles = full; b.row_tiles = w.row_tiles - full;
    pick_tile(BAMD_ACT_BF16, w, rows, 1, share, out, &whole);
    const int ta = pick_tile(BAMD_ACT_BF16, a, rows, 1, share, out, &ca);
    pick_tile(BAMD_ACT_BF16, b, rows, 1, share, out, &cb);
    return ta == TILE_256_256 && (ca + cb + 4000) * 103 < whole * 100 ? full : 0;
}
template <typename T, int OUT>
static int gemm_tiles(const bamd_dense & w, const void * x, int ldx, int cb, int rows, void * out, int ldo, int cbo, float limit, hipStream_t s, int * parts = nullptr) {
    int share;
    const int tile = pick_tile(sizeof(T) == 4 ? BAMD_ACT_F32 : BAMD_ACT_BF16, w, rows, OUT == BAMD_OUT_F32 && parts ? *parts : 1, share, OUT);
    if (parts) *parts = share;
    if constexpr (sizeof(T) == 2 && (OUT == BAMD_OUT_F32 || OUT == BAMD_OUT_GLU)) if (const int n = share == 1 ? bamd_dense_cut(w, rows, OUT) : 0) {
        bamd_dense a = w, b = w;
        a.row_tiles = n; a.rows = std::min(w.rows, n * 16);
        b.row_tiles = w.row_tiles - n; b.rows = w.rows - n * 16; b.w = w.w + (size_t) n * w.k_tiles * 512;
        void * rest = OUT == BAMD_OUT_F32 ? (void *) ((float *) out + n * 16) : (T *) out + (cbo ? (size_t) (n / 4) * cbo : (size_t) n * 8);
        return gemm_tiles<T, OUT>(a, x, ldx, cb, rows, out, ldo, cbo, limit, s) || gemm_tiles<T, OUT>(b, x, ldx, cb, rows, rest, ldo, cbo, limit, s);
    }
    if constexpr (sizeof(T) == 2) switch (tile) {
        case TILE_256_256: return tile_go<T, 256, 256, 2, 4, 4, OUT>(w, x, ldx, cb, rows, out, ldo, cbo, limit, share, s);
        case TILE_256_224: if constexpr (OUT != BAMD_OUT_GLU) return tile_go<T, 256, 224, 4, 2, 4, OUT>(w, x, ldx, cb, rows, out, ldo, cbo, limit, share, s); else return 1;
        case TILE_256_192: return tile_go<T, 256, 192, 4, 2, 4, OUT>(w, x, ldx, cb, rows, out, ldo, cbo, limit, share, s);
        case TILE_256_160: if constexpr (OUT != BAMD_OUT_GLU) return tile_go<T, 256, 160, 4, 2, 4, OUT>(w, x, ldx, cb, rows, out, ldo, cbo, limit, share, s); else return 1;
        case TILE_128_256: return tile_go<T, 128, 256, 2, 4, 4, OUT>(w, x, ldx, cb, rows, out, ldo, cbo, limit, share, s);
        case TILE_128_128: return tile_go<T, 128, 128, 2, 4, 8, OUT>(w, x, ldx, cb, rows, out, ldo, cbo, limit, share, s);
        case TILE_64_128: return tile_go<T, 64, 128, 2, 2, 4, OUT>(w, x, ldx, cb, rows, out, ldo, cbo, limit, share, s);
        case TILE_64_64_DEEP: return tile_go<T, 64, 64, 2, 2, 8, OUT>(w, x, ldx, cb, rows, out, ldo, cbo, limit, share, s);
    }
    else switch (tile) {                                          // three planes of activations: waves as tall as wide would read twice as much of them
        case TILE_128_256: return tile_go<T, 128, 256, 2, 4, 4, OUT>(w, x, ldx, cb, rows, out, ldo, cbo, limit, share, s);
        case TILE_128_128: return tile_go<T, 128, 128, 4, 2, 4, OUT>(w, x, ldx, cb, rows, out, ldo, cbo, limit, share, s);
        case TILE_64_128: return tile_go<T, 64, 128, 2, 2, 4, OUT>(w, x, ldx, cb, rows, out, ldo, cbo, limit, share, s);
    }
    return tile_go<T, 64, 64, 2, 2, 4, OUT>(w, x, ldx, cb, rows, out, ldo, cbo, limit, share, s);
}
// operand rows start on 16 bytes and hold k_tiles * 32 columns, or lie by blocks
static bool rows_fit(const bamd_dense & w, int ldx, int cb, int rows, int in_block) { return cb ? cb >= in_block * rows && !(cb & 7) : ldx >= w.k_tiles * in_block && !(ldx & 7); }
// f32 rows are stored four matrix rows at a time: ldo % 4 == 0
template <typename T>
static int gemm_out(const bamd_dense & w, const void * x, int ldx, int cb, int rows, void * out, int ldo, int cbo, int kind, float limit, hipStream_t s, int * parts) {
    if (kind != BAMD_OUT_F32 && parts) *parts = 1;
    switch (kind) {
        case BAMD_OUT_F32: return gemm_tiles<T, BAMD_OUT_F32>(w, x, ldx, cb, rows, out, ldo, 0, limit, s, parts);
        case BAMD_OUT_ACT: return gemm_tiles<T, BAMD_OUT_ACT>(w, x, ldx, cb, rows, out, ldo, 0, limit, s);
        case BAMD_OUT_ACT_T: return gemm_tiles<T, BAMD_OUT_ACT_T>(w, x, ldx, cb, rows, out, ldo, 0, limit, s);
        case BAMD_OUT_GLU: return (w.row_tiles & 1) || ldo < w.row_tiles * 8 ? 1 : gemm_tiles<T, BAMD_OUT_GLU>(w, x, ldx, cb, rows, out, ldo, cbo, limit, s);
    }
    return 1;
}
int bamd_launch_dense_gemm(int act, const bamd_dense & w, const void * x, int ldx, int cb, int rows, void * out, int ldo, int kind, hipStream_t s, float limit, int * parts, int cbo) {
    const int in_block = 32 * bamd_row_planes(act);
    if (rows < 1 || w.row_tiles < 1 || w.k_tiles < 1 || (ldo & 3) || !rows_fit(w, ldx, cb, rows, in_block)) return 1;
    if (cb) ldx = in_block; else cb = in_block;
    return act == BAMD_ACT_F32 ? gemm_out<float>(w, x, ldx, cb, rows, out, ldo, cbo, kind, limit, s, parts) : gemm_out<bamd_bf>(w, x, ldx, cb, rows, out, ldo, cbo, kind, limit, s, parts);
}

// ---- few rows ---------------------------------------------------------------------------------------------------------------------------------------
// NT: groups of 16 rows; NW: waves; U: 32-column blocks per request batch of a wave
// where a lane's four sums lie among a wave's 256: sixteen lanes that read four outputs each, of four rows, find them in different banks
__device__ __forceinline__ int sum_slot(int l) { return ((l & 48) | ((l ^ (l >> 2 & 12)) & 15)) * 4; }
// The last product of a decoding step brings its results to the host as it goes (stores that write through, 64 bytes of a row per instruction: in pieces of eight a row of 32 000 takes 1.3 ms)
// and says when they are there: every wave waits for its own, the block that is done last tells the host.  The count itself orders nothing (acquire and release at every block's end are
// write-backs of the L2: 10 us of a step).  A launch behind the product took 50 us for sixteen rows of 32 000, 6.5 for one; a step of eight layers, width 2048, one row 437 -> 430 us, six rows 649 ->
// 632, width 4096, sixteen rows 1333 -> 1304, 32-bit, eight rows 808 -> 776
__device__ __forceinline__ void to_host(const bamd_step_out & c, size_t at, float v) { if (c.host) __hip_atomic_store(c.host + at, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM); }
__device__ __forceinline__ void close_step(const bamd_step_out & c) {
    if (!c.count_serial) return;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x || __hip_atomic_fetch_add(c.count_serial, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1 < gridDim.x * gridDim.y) return;
    c.count_serial[0] = 0;
    __threadfence_system();
    __hip_atomic_store(c.done, c.count_serial[1], __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}
template <typename T, int NT, int NW, int PRE, bool ONE>
__global__ void __launch_bounds__(64 * NW) dense_mv_kernel(bamd_dense w, bamd_batch_dev b, bamd_pre_args p, const bamd_bf * x, int ldx, int cb, int rows, float * out, int ldo) {
    constexpr int U = 8, P = bamd_planes<T>;
    typedef Operand<T> O;
    extern __shared__ __align__(16) unsigned char lds[];
    __shared__ float red[NW * NT * 256];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int kb = w.k_tiles * blockIdx.y / gridDim.y, ke = w.k_tiles * (blockIdx.y + 1) / gridDim.y;      // the block's share of K, and the wave's
    const int k0 = kb + (ke - kb) * wave / NW, k1 = kb + (ke - kb) * (wave + 1) / NW, kn = (ke - kb + NW - 1) / NW, nc = (kn + U - 1) / U;
    out += (size_t) blockIdx.y * rows * ldo;
    bamd_u4 cur[U], nxt[U] = {};
    auto request = [&](int tile, int c, bamd_u4 * d) {
        const uint16_t * base = w.w + ((size_t) tile * w.k_tiles * 64 + lane) * 8;
#pragma unroll
        for (int u = 0; u < U; ++u) { int kt = k0 + c * U + u; kt = kt < w.k_tiles ? kt : w.k_tiles - 1; d[u] = *(const bamd_u4 *) (base + (size_t) kt * 512); }
    };
    int tile = blockIdx.x;
    request(tile, 0, cur);                                        // on their way while the operand row is built
    if constexpr (PRE != BAMD_PRE_ROWS) {
        const RowOut<O> h = { (O *) lds, 32 * P };
        if constexpr (PRE == BAMD_PRE_RESIDUAL) residual_row<O, true, ONE>(b, p.res, 0, h, blockIdx.x == 0, red);
        if constexpr (PRE == BAMD_PRE_POLY) poly_row<O, ONE>(p.poly, 0, h, red);
        if constexpr (PRE == BAMD_PRE_GROUP) group_norm_row<O>(p.grp, 0, h, red);
        if constexpr (PRE == BAMD_PRE_GLU) glu_row<O>(p.glu, 0, h, 0, p.glu.ldh);
        if constexpr (PRE == BAMD_PRE_LAYER) layer_row<O, ONE>(p.res, p.want ? p.want[0] : 0, p.want ? p.gf : p.res.gi, h, !p.want && blockIdx.x == 0, red);
        if constexpr (PRE == BAMD_PRE_FINAL) final_row<O, ONE>(p.res, p.want[0], p.gf, h, red);
        __syncthreads();
    }
    const int col = lane & 15, kq = (lane >> 4) * 8;
    for (; tile < w.row_tiles; tile += gridDim.x) {
        bamd_v4 acc[NT];
#pragma unroll
        for (int n = 0; n < NT; ++n) acc[n] = bamd_v4{ 0, 0, 0, 0 };
        for (int c = 0; c < nc; ++c) {
            const bool more = c + 1 < nc;
            if (more) request(tile, c + 1, nxt);
            else if (tile + (int) gridDim.x < w.row_tiles) request(tile + gridDim.x, 0, nxt);
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int kt = k0 + c * U + u;
                if (kt < k1) {
                    const bamd_bf8 wf = __builtin_bit_cast(bamd_bf8, cur[u]);
#pragma unroll
                    for (int n = 0; n < NT; ++n) {
                        const bamd_bf * at;
                        if constexpr (PRE != BAMD_PRE_ROWS) at = (const bamd_bf *) lds + kt * (32 * P) + kq;
                        else { int r = n * 16 + col; r = r < rows ? r : rows - 1; at = x + (size_t) r * ldx + (size_t) kt * cb + kq; }
                        if constexpr (P == 1) acc[n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf, *(const bamd_bf8 *) at, acc[n], 0, 0, 0);
                        else {                                    // (from zero, and added by the vector units: dense_tile_kernel)
                            bamd_v4 s = { 0, 0, 0, 0 };
#pragma unroll
                            for (int i = P - 1; i >= 0; --i) s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf, *(const bamd_bf8 *) (at + i * 32), s, 0, 0, 0);
                            acc[n] = acc[n] + s;
                        }
                    }
                }
            }
#pragma unroll
            for (int u = 0; u < U; ++u) cur[u] = nxt[u];
        }
        __syncthreads();                                          // (the sums of the tile before are read)
#pragma unroll
        for (int n = 0; n < NT; ++n) *(bamd_v4 *) (red + (wave * NT + n) * 256 + sum_slot(lane)) = acc[n];
        __syncthreads();
        for (int i = tid; i < NT * 256; i += 64 * NW) {           // sixteen outputs of a row per sixteen lanes: four each, on a quarter of the lanes, are 1 to 2 % of a step slower
            const int n = i >> 8, c = i & 15, rl = (i >> 4) & 15, r = n * 16 + rl, o = tile * 16 + c;
            if (r < rows && o < w.rows) {
                float v = 0.f;
#pragma unroll
                for (int q = 0; q < NW; ++q) v += red[(q * NT + n) * 256 + sum_slot((c >> 2) * 16 + rl) + (c & 3)];
                out[(size_t) r * ldo + o] = v;
                to_host(p.close, (size_t) r * ldo + o, v);
            }
        }
    }
    close_step(p.close);
}
// Up to 64 rows, bfloat16: NT groups of 16 rows, RT row tiles of the matrix.  Every block reads all the rows: bytes out of L2 (NT per RT of weights) and, read by the lanes of a
// fragment as above, four times the lookups of the same bytes in one piece, were what the product took (16 rows x 14336 x 4096: 32 us, of which the weights are 19).  Here every
// wave streams its share of K — RT KiB of weights and NT of the rows per step — by DMA through a ring of NS steps of its own: 64 consecutive bytes of a row per four lanes, read
// back in fragment order (dense_tile_kernel's layout), no barrier between steps, and while the sums of a group of tiles meet, the next group's first steps are under way.  LDS holds
// one block of eight waves per CU.  16 x 14336 x 4096: 32.3 -> 27.1 us (4.3 TB/s of weights), 16 x 32000 x 4096: 62 -> 50 (5.3), 45 x 4096 x 14336: 57 -> 48 us.
// Rows by blocks (bamd_dense.h): a step of eight layers, sixteen rows 1390 -> 1318 us (width 4096), 835 -> 817 (2048), 32 rows 1918 -> 1737 and 1226 -> 1143, 64 rows 2772 -> 2493 and 1716 -> 1573; up to six
// rows, where the few there are cost little, level.
// GLU (an even RT): gate and up tiles in turn; out is the gated unit's bfloat16 row.
template <int NT, int RT, int NS, bool GLU>
__global__ void __launch_bounds__(512) dense_few_kernel(bamd_dense w, const bamd_bf * x, int ldx, int cb, int rows, float * out, int ldo, int cbo, float limit, bamd_step_out close) {
    constexpr int NW = 8, STEP = (NT + RT) * 1024, RING = NS * STEP;
    extern __shared__ __align__(16) unsigned char lds[];
    float * red = (float *) (lds + NW * RING);                    // [wave][RT][NT][64 lanes][4]
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kb = w.k_tiles * blockIdx.y / gridDim.y, ke = w.k_tiles * (blockIdx.y + 1) / gridDim.y, k0 = kb + (ke - kb) * wave / NW, n = kb + (ke - kb) * (wave + 1) / NW - k0;      // the block's share of K, and the wave's
    const int groups = (w.row_tiles + RT - 1) / RT;
    out += (size_t) blockIdx.y * rows * ldo;
    uint32_t xo[NT];
#pragma unroll
    for (int g = 0; g < NT; ++g) { int r = g * 16 + (lane >> 2); r = r < rows ? r : rows - 1; xo[g] = (uint32_t) r * (uint32_t) ldx * 2u + (uint32_t) ((lane & 3) ^ ((lane >> 3) & 3)) * 16u; }
    const uint32_t ring = (uint32_t) (size_t) (bamd_lds_vp) lds + (uint32_t) wave * RING;
    const unsigned char * mine = lds + (size_t) wave * RING, * xs = mine + 1024 * RT + ((lane & 15) * 4 + ((lane >> 4) ^ ((lane >> 1) & 3))) * 16;
    int ct = blockIdx.x, ck = 0, cs = 0;                          // next copy: group of RT row tiles, step, slot
    auto copy = [&] {                                             // (behind the last step: its bytes again, into slots nobody reads)
        const size_t k = (size_t) (k0 + ck);
#pragma unroll
        for (int t = 0; t < RT; ++t) {
            int tile = ct * RT + t; tile = tile < w.row_tiles ? tile : w.row_tiles - 1;
            lds_dma16_s(w.w + ((size_t) tile * w.k_tiles + k) * 512, (uint32_t) lane * 16u, ring + (uint32_t) cs * STEP + 1024u * t);
        }
#pragma unroll
        for (int g = 0; g < NT; ++g) lds_dma16_s((const unsigned char *) x + k * cb * 2, xo[g], ring + (uint32_t) cs * STEP + 1024u * (g + RT));
        cs = cs + 1 < NS ? cs + 1 : 0;
        if (ck + 1 < n) ++ck; else if (ct + (int) gridDim.x < groups) { ck = 0; ct += gridDim.x; }
    };
    if (n > 0)
        for (int i = 0; i < NS - 1; ++i) copy();
    int slot = 0;
    for (int grp = blockIdx.x; grp < groups; grp += gridDim.x) {
        bamd_v4 acc[RT][NT];
#pragma unroll
        for (int t = 0; t < RT; ++t)
#pragma unroll
            for (int g = 0; g < NT; ++g) acc[t][g] = bamd_v4{ 0, 0, 0, 0 };
        for (int i = 0; i < n; ++i) {
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" :: "n"((NS - 2) * (NT + RT)) : "memory");      // this step has landed; the step before is read
            copy();
            const int at = slot * STEP;
            slot = slot + 1 < NS ? slot + 1 : 0;
            bamd_bf8 wf[RT], xf[NT];
#pragma unroll
            for (int t = 0; t < RT; ++t) wf[t] = *(const bamd_bf8 *) (mine + at + t * 1024 + lane * 16);
#pragma unroll
            for (int g = 0; g < NT; ++g) xf[g] = *(const bamd_bf8 *) (xs + at + g * 1024);
#pragma unroll
            for (int t = 0; t < RT; ++t)
#pragma unroll
                for (int g = 0; g < NT; ++g) acc[t][g] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[t], xf[g], acc[t][g], 0, 0, 0);
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();                             // (the sums of the tiles before are read)
        asm volatile("" ::: "memory");
#pragma unroll
        for (int t = 0; t < RT; ++t)
#pragma unroll
            for (int g = 0; g < NT; ++g) *(bamd_v4 *) (red + ((wave * RT + t) * NT + g) * 256 + sum_slot(lane)) = acc[t][g];
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        auto sum = [&](int c, int rl, int o) {                    // of column o, row rl of cell c
            float v = 0.f;
#pragma unroll
            for (int q = 0; q < NW; ++q) v += red[(q * RT * NT + c) * 256 + sum_slot((o >> 2) * 16 + rl) + (o & 3)];
            return v;
        };
        if constexpr (GLU) {
            for (int i = tid; i < RT / 2 * NT * 256; i += 64 * NW) {
                const int c = i >> 8, t = c / NT * 2, oc = i & 15, rl = (i >> 4) & 15, r = (c % NT) * 16 + rl, o = (grp * RT + t) * 8 + oc;
                if (r < rows && o < w.rows / 2) *row_out<bamd_bf>(out, r, ldo, cbo).at(o) = (bamd_bf) clamped_glu(sum(t * NT + c % NT, rl, oc), sum((t + 1) * NT + c % NT, rl, oc), limit);
            }
        } else for (int i = tid; i < RT * NT * 256; i += 64 * NW) {
            const int c = i >> 8, oc = i & 15, rl = (i >> 4) & 15, r = (c % NT) * 16 + rl, o = (grp * RT + c / NT) * 16 + oc;
            if (r < rows && o < w.rows) {
                const float v = sum(c, rl, oc);
                out[(size_t) r * ldo + o] = v;
                to_host(close, (size_t) r * ldo + o, v);
            }
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");              // (no copy outlives the block)
    close_step(close);
}
template <int NT, int RT, int NS, bool GLU = false>
static void few_go(const bamd_dense & w, const void * x, int ldx, int cb, int rows, float * out, int ldo, hipStream_t s, int parts, const bamd_step_out & close, int cbo = 0, float limit = 0.f) {
    const int groups = (w.row_tiles + RT - 1) / RT;
    hipLaunchKernelGGL((dense_few_kernel<NT, RT, NS, GLU>), dim3(groups < 256 ? groups : 256, parts), dim3(512), (size_t) 8 * (NS * (NT + RT) + NT * RT) * 1024, s, w, (const bamd_bf *) x, ldx, cb, rows, out, ldo, cbo, limit, close);
}
// The same for up to sixteen rows where a block has several row tiles to go through and the rows' shares of K fit LDS: each wave copies its share of the rows once, in front of the loop, and its weights
// go straight to registers, D requests of a kilobyte ahead, from one tile into the next.  Tiles are dealt out one by one (GLU: in pairs of gate and up), so that no CU has more than one above the
// others — dense_few_kernel's groups of two or three leave up to a third of a round idle — and neighbours read neighbouring memory (a run of tiles per block: up to 18 % slower where the runs lie half a
// megabyte apart).  The weights are requested first and everything is waited for once: rows first were 1 to 4 % slower.  Eight requests ahead: 1 to 6 % slower, sixteen: level.  Sums of up to `meet` tiles
// wait in LDS for the eight waves to meet; they are the sums of dense_few_kernel, in its order.  us, that kernel and this one, behind a launch that writes the rows (its 2 us included): 16 rows x 14336 x
// 4096 27.7 | 24.2 (5.2 TB/s), 16768 x 4096 32.8 | 28.5, 32000 x 4096 52.2 | 47.8, 28672 x 4096 with the gated unit 49.1 | 44.6, two rows x 8192 x 4096 18.1 | 15.8.
template <int D, bool GLU>
__global__ void __launch_bounds__(512) dense_share_kernel(bamd_dense w, const bamd_bf * x, int ldx, int cb, int rows, float * out, int ldo, int cbo, float limit, bamd_step_out close, int meet) {
    constexpr int NW = 8, UNIT = GLU ? 2 : 1;
    extern __shared__ __align__(16) unsigned char lds[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), stride = gridDim.x;
    const int k0 = w.k_tiles * wave / NW, n = w.k_tiles * (wave + 1) / NW - k0, kn = (w.k_tiles + NW - 1) / NW;
    float * red = (float *) (lds + (size_t) NW * kn * 1024);       // [wave][meet][64 lanes][4], behind the rows
    const int tiles = (w.row_tiles / UNIT - (int) blockIdx.x + stride - 1) / stride * UNIT, steps = tiles * n;
    auto tile_of = [&](int j) { return ((int) blockIdx.x + j / UNIT * stride) * UNIT + j % UNIT; };
    const uint16_t * src = w.w + ((size_t) tile_of(0) * w.k_tiles + k0) * 512;
    const size_t near = (size_t) (w.k_tiles - n + 1) * 512, far = near + (size_t) (stride - 1) * UNIT * w.k_tiles * 512;      // from a share's end to the next tile's
    int rk = 0, rj = 0, left = steps;
    bamd_u4 ring[D];
    auto request = [&](int u) {                                   // (behind the last step: that one again, for nobody)
        ring[u] = *(const bamd_u4 *) (src + lane * 8);
        if (--left > 0) { if (++rk < n) src += 512; else { rk = 0; ++rj; src += GLU && (rj & 1) ? near : far; } }
    };
#pragma unroll
    for (int u = 0; u < D; ++u) request(u);
    {
        int r = lane >> 2; r = r < rows ? r : rows - 1;
        const uint32_t xo = (uint32_t) r * (uint32_t) ldx * 2u + (uint32_t) ((lane & 3) ^ ((lane >> 3) & 3)) * 16u, to = (uint32_t) (size_t) (bamd_lds_vp) lds + (uint32_t) (wave * kn) * 1024u;
        for (int k = 0; k < n; ++k) lds_dma16_s((const unsigned char *) x + (size_t) (k0 + k) * cb * 2, xo, to + (uint32_t) k * 1024u);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    const unsigned char * xs = lds + (size_t) wave * kn * 1024 + ((lane & 15) * 4 + ((lane >> 4) ^ ((lane >> 1) & 3))) * 16;
    bamd_v4 acc = { 0, 0, 0, 0 };
    int k = 0, waiting = 0, first = 0;                             // tiles whose sums wait; the first of them
    auto all_here = [&] { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); __builtin_amdgcn_s_barrier(); asm volatile("" ::: "memory"); };
    auto join = [&](int count) {
        all_here();
        auto sum = [&](int t, int rl, int o) {                    // of column o, row rl of tile t
            float v = 0.f;
#pragma unroll
            for (int q = 0; q < NW; ++q) v += red[(q * meet + t) * 256 + sum_slot((o >> 2) * 16 + rl) + (o & 3)];
            return v;
        };
        for (int i = tid; i < count / UNIT * 256; i += 64 * NW) {
            const int t = (i >> 8) * UNIT, oc = i & 15, r = (i >> 4) & 15, o = tile_of(first + t) / UNIT * 16 + oc;
            if (r >= rows || o >= w.rows / UNIT) continue;
            if constexpr (GLU) *row_out<bamd_bf>(out, r, ldo, cbo).at(o) = (bamd_bf) clamped_glu(sum(t, r, oc), sum(t + 1, r, oc), limit);
            else {
                const float v = sum(t, r, oc);
                out[(size_t) r * ldo + o] = v;
                to_host(close, (size_t) r * ldo + o, v);
            }
        }
        first += count;
    };
    auto take = [&](int u) {
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bamd_bf8, ring[u]), *(const bamd_bf8 *) (xs + k * 1024), acc, 0, 0, 0);
        if (++k < n) return;
        *(bamd_v4 *) (red + (wave * meet + waiting) * 256 + sum_slot(lane)) = acc;
        acc = bamd_v4{ 0, 0, 0, 0 }; k = 0;
        if (++waiting == meet) { join(meet); waiting = 0; all_here(); }      // (every wave has as many tiles, and at least a column block of each)
    };
    int s = 0;
    for (; s + D <= steps; s += D)
#pragma unroll
        for (int u = 0; u < D; ++u) { take(u); request(u); }
#pragma unroll
    for (int u = 0; u < D; ++u) if (s + u < steps) take(u);
    if (waiting) join(waiting);
    close_step(close);
}
// Where whole decoding steps are ahead, dense_few_kernel and this one, us, four layers each: width 4096 (Tupitar) two rows 562 | 546, sixteen 855 | 822; (Mafurax) six rows 793 | 775; width 3200,
// thirteen rows 602 | 600; 3584, three rows 548 | 546.  Below K = 3072 the products by themselves are ahead (11328 x 2048 6 % at two rows), steps are not: width 2048, six rows 367 | 367, width 1024, twelve
// rows 238 | 240.  With two tiles a block it takes K of about 4096 (two rows x 4640 x 3072 10.7 | 10.9, x 4096 13.1 | 12.4, x 4608 11.2 | 11.8), and K beyond 4608 leaves no room for the sums
static bool share_fits(const bamd_dense & w, int rows) {
    if (rows > 16 || w.k_tiles < 96 || w.k_tiles > 144) return false;
    return w.row_tiles > 512 || (w.row_tiles > 256 && w.k_tiles >= 112 && w.k_tiles <= 128);
}
template <bool GLU>
static void share_go(const bamd_dense & w, const void * x, int ldx, int cb, int rows, float * out, int ldo, hipStream_t s, const bamd_step_out & close, int cbo = 0, float limit = 0.f) {
    constexpr int unit = GLU ? 2 : 1;
    const int units = w.row_tiles / unit, grid = units < 256 ? units : 256, kn = (w.k_tiles + 7) / 8, most = (units + grid - 1) / grid * unit;
    // A product that brings its results to the host meets after every tile: the bus is slower than the sums, and with eight tiles together all of them waited for it at the end (six rows of 32000: 31 | 40 us)
    const int meet = close.host ? 1 : std::min(most, (20 - kn) / unit * unit);      // of 160 KiB, eight a tile
    const size_t lds = (size_t) 8 * (kn + meet) * 1024;
    hipLaunchKernelGGL((dense_share_kernel<12, GLU>), dim3(grid), dim3(512), lds, s, w, (const bamd_bf *) x, ldx, cb, rows, out, ldo, cbo, limit, close, meet);
}
bool bamd_dense_closes(int act, const bamd_dense & w, int rows, int ldo) { return act == BAMD_ACT_F32 || rows <= 32 || w.row_tiles <= 768 || (ldo & 3); }
// RT by the rounds over the CUs; a round of 1, 2 or 3 tiles at K = 4096 takes 7.1, 12.7 and 16 us with up to 16 rows, one of 1 or 2 tiles 9.0 and 15.1 us with up to 32.
// With more rows the 64 x 64 tiles of prompts are ahead once they fill the CUs (45 x 22672 x 4096: 49 against 74 us) and behind before (45 x 4096 x 14336: 136 against 48)
static int few_pick(const bamd_dense & w, const void * x, int ldx, int cb, int rows, float * out, int ldo, hipStream_t s, int parts, const bamd_step_out & close) {
    const long rounds[3] = { (w.row_tiles + 255) / 256, (w.row_tiles + 511) / 512, (w.row_tiles + 767) / 768 };
    if (rows > 32) {
        if (!bamd_dense_closes(BAMD_ACT_BF16, w, rows, ldo)) return gemm_tiles<bamd_bf, BAMD_OUT_F32>(w, x, ldx, cb, rows, out, ldo, 0, 0.f, s);
        few_go<4, 1, 3>(w, x, ldx, cb, rows, out, ldo, s, parts, close);
    } else if (rows > 16) {
        if (rounds[0] * 90 <= rounds[1] * 151) few_go<2, 1, 5>(w, x, ldx, cb, rows, out, ldo, s, parts, close); else few_go<2, 2, 4>(w, x, ldx, cb, rows, out, ldo, s, 1, close);
    } else if (share_fits(w, rows)) share_go<false>(w, x, ldx, cb, rows, out, ldo, s, close);
    else {
        const long t1 = rounds[0] * 71, t2 = rounds[1] * 127, t3 = rounds[2] * 160;
        if (t1 <= t2 && t1 <= t3) few_go<1, 1, 5>(w, x, ldx, cb, rows, out, ldo, s, parts, close);
        else if (t2 <= t3) few_go<1, 2, 5>(w, x, ldx, cb, rows, out, ldo, s, 1, close);
        else few_go<1, 3, 4>(w, x, ldx, cb, rows, out, ldo, s, 1, close);
    }
    return 0;
}
size_t bamd_dense_mv_lds(int act, int K) { return (size_t) (K + 31) / 32 * 64 * bamd_row_planes(act); }
template <typename T, int NT, int NW, int PRE>
static void mv_go(const bamd_dense & w, const bamd_batch_dev & b, const bamd_pre_args & p, const void * x, int ldx, int cb, int n, float * out, int ldo, hipStream_t s, int parts = 1) {
    const int grid = w.row_tiles < 4096 / NW ? w.row_tiles : 4096 / NW;       // what is resident at once; blocks walk the tiles
    const size_t lds = PRE == BAMD_PRE_ROWS ? 0 : bamd_dense_mv_lds(sizeof(T) == 4 ? BAMD_ACT_F32 : BAMD_ACT_BF16, w.k_tiles * 32);
    constexpr bool rows = PRE == BAMD_PRE_RESIDUAL || PRE == BAMD_PRE_LAYER || PRE == BAMD_PRE_FINAL;
    if constexpr (rows || PRE == BAMD_PRE_POLY)
        if ((rows ? p.res.E : p.poly.F) & 3) { hipLaunchKernelGGL((dense_mv_kernel<T, NT, NW, PRE, true>), dim3(grid, parts), dim3(64 * NW), lds, s, w, b, p, (const bamd_bf *) x, ldx, cb, n, out, ldo); return; }
    hipLaunchKernelGGL((dense_mv_kernel<T, NT, NW, PRE, false>), dim3(grid, parts), dim3(64 * NW), lds, s, w, b, p, (const bamd_bf *) x, ldx, cb, n, out, ldo);
}
// sixteen waves where the tiles alone would leave the chip half empty
template <typename T, int PRE>
static void mv_one(const bamd_dense & w, const bamd_batch_dev & b, const bamd_pre_args & p, const void * x, int ldx, int cb, int rows, float * out, int ldo, hipStream_t s, int parts = 1) {
    if (w.row_tiles <= 256) mv_go<T, 1, 16, PRE>(w, b, p, x, ldx, cb, rows, out, ldo, s, parts);
    else mv_go<T, 1, 8, PRE>(w, b, p, x, ldx, cb, rows, out, ldo, s);
}
// Two shares of K where a matrix has too few row tiles for the CUs (more than 128 would make a second round of their blocks) and enough columns that halves are still worth a block: at K = 2048
// they are level with 8 rows (2048 outputs: 5.7 us) and ahead with more (45 rows 8.7 -> 7.5) or longer rows (K = 4096: 7.1 -> 6.5, 11.8 -> 9.4).  A prologue that writes state stays whole.  A bfloat16
// row built in front is built whole by either half's block, which more than 64 row tiles pay back where the whole product's waves would need a second round of eight column blocks, beyond K = 4096
// (1536 outputs, PolyNorm: K = 4096 8.8 us whole, 9.2 in halves; 4128 9.6 and 9.2; 64 row tiles: 8.7 and 8.7); the 32-bit products behind it are longer (12.5 and 11.5)
static int few_parts(int act, const bamd_dense & w, int pre, int most) {
    if (most < 2 || w.row_tiles > 128 || w.k_tiles < 64 || pre == BAMD_PRE_RESIDUAL || pre == BAMD_PRE_FINAL || pre == BAMD_PRE_LAYER) return 1;
    return act == BAMD_ACT_BF16 && pre != BAMD_PRE_ROWS && w.row_tiles > 64 && w.k_tiles <= 128 ? 1 : 2;
}
int bamd_dense_route(int act, const bamd_dense & w, int rows, int pre, int most, int & share) {
    if (pre < 0) return pick_tile(act, w, rows, most, share, BAMD_OUT_F32);
    share = few_parts(act, w, pre, most);
    return -1;
}
template <typename T>
static int mv_pick(const bamd_dense & w, int pre, const bamd_batch_dev & b, const bamd_pre_args & p, const void * x, int ldx, int cb, int rows, float * out, int ldo, hipStream_t s, int * parts) {
    const int n = few_parts(sizeof(T) == 4 ? BAMD_ACT_F32 : BAMD_ACT_BF16, w, pre, parts ? *parts : 1);
    if (parts) *parts = n;
    if (pre != BAMD_PRE_ROWS) {
        if (rows != 1 || bamd_dense_mv_lds(sizeof(T) == 4 ? BAMD_ACT_F32 : BAMD_ACT_BF16, w.k_tiles * 32) > BAMD_MV_LDS(sizeof(T) == 4 ? BAMD_ACT_F32 : BAMD_ACT_BF16)) return 1;
        const int ldh = pre == BAMD_PRE_POLY ? p.poly.ldh : pre == BAMD_PRE_GROUP ? p.grp.ldh : pre == BAMD_PRE_GLU ? p.glu.ldh : p.res.ldh;
        if (ldh != w.k_tiles * 32) return 1;
        if (pre == BAMD_PRE_RESIDUAL && p.res.norm != BAMD_NORM_LAYER) mv_one<T, BAMD_PRE_RESIDUAL>(w, b, p, x, ldx, cb, rows, out, ldo, s);
        else if (pre == BAMD_PRE_POLY) mv_one<T, BAMD_PRE_POLY>(w, b, p, x, ldx, cb, rows, out, ldo, s, n);
        else if (pre == BAMD_PRE_GROUP) mv_one<T, BAMD_PRE_GROUP>(w, b, p, x, ldx, cb, rows, out, ldo, s, n);
        else if (pre == BAMD_PRE_GLU) mv_one<T, BAMD_PRE_GLU>(w, b, p, x, ldx, cb, rows, out, ldo, s, n);
        else if (p.res.norm == BAMD_NORM_LAYER) mv_one<T, BAMD_PRE_LAYER>(w, b, p, x, ldx, cb, rows, out, ldo, s);
        else mv_one<T, BAMD_PRE_FINAL>(w, b, p, x, ldx, cb, rows, out, ldo, s);
        return 0;
    }
    const int in_block = 32 * bamd_planes<T>;
    if (rows < 1 || rows > BAMD_MV_ROWS || !rows_fit(w, ldx, cb, rows, in_block)) return 1;
    if (cb) ldx = in_block; else cb = in_block;
    if constexpr (sizeof(T) == 2) return few_pick(w, x, ldx, cb, rows, out, ldo, s, n, p.close);
    else if (rows <= 16) mv_one<T, BAMD_PRE_ROWS>(w, b, p, x, ldx, cb, rows, out, ldo, s, n);
    else if (rows <= 32) mv_go<T, 2, 8, BAMD_PRE_ROWS>(w, b, p, x, ldx, cb, rows, out, ldo, s, n);
    else mv_go<T, 4, 8, BAMD_PRE_ROWS>(w, b, p, x, ldx, cb, rows, out, ldo, s, n);
    return 0;
}
// The gated unit as a part of the product in front of it costs the launch behind that (4 us) and 32-bit results on their way through memory; it asks for pairs of row tiles, which a block of
// up to 32 rows has where it takes two.  A decoding step of 8 layers, before and after: 2048 x 16384 6 rows 675 -> 657 us, 16 866 -> 848, 17 931 -> 897; 4096 x 28672 (three tiles a block were ahead
// without) 6 rows 1368 -> 1350, 16 1683 -> 1660.  Four tiles a block: 666, 848; 1394, 1684.  More rows: where few_pick takes the tiles of prompts, they have the unit as well
// (64 rows 3181 -> 3141)
bool bamd_dense_few_glu(int act, const bamd_dense & w, int rows) { return act == BAMD_ACT_BF16 && !(w.row_tiles & 1) && rows > 1 && (rows <= 32 || (rows <= BAMD_MV_ROWS && w.row_tiles > 768)); }
int bamd_launch_dense_few_glu(const bamd_dense & w, const void * x, int ldx, int cb, int rows, void * h, int ldh, int cbo, float limit, hipStream_t s) {
    if (!bamd_dense_few_glu(BAMD_ACT_BF16, w, rows) || !rows_fit(w, ldx, cb, rows, 32) || ldh < w.row_tiles * 8 || (ldh & 3)) return 1;
    if (cb) ldx = 32; else cb = 32;
    if (rows > 32) return gemm_tiles<bamd_bf, BAMD_OUT_GLU>(w, x, ldx, cb, rows, h, ldh, cbo, limit, s);
    if (rows > 16) few_go<2, 2, 4, true>(w, x, ldx, cb, rows, (float *) h, ldh, s, 1, {}, cbo, limit);
    else if (share_fits(w, rows)) share_go<true>(w, x, ldx, cb, rows, (float *) h, ldh, s, {}, cbo, limit);
    else few_go<1, 2, 5, true>(w, x, ldx, cb, rows, (float *) h, ldh, s, 1, {}, cbo, limit);
    return 0;
}
int bamd_launch_dense_mv(int act, const bamd_dense & w, int pre, const bamd_batch_dev & b, const bamd_pre_args * p, const void * x, int ldx, int cb, int rows, float * out, int ldo, hipStream_t s, int * parts) {
    static const bamd_pre_args none = {};
    return act == BAMD_ACT_F32 ? mv_pick<float>(w, pre, b, p ? *p : none, x, ldx, cb, rows, out, ldo, s, parts) : mv_pick<bamd_bf>(w, pre, b, p ? *p : none, x, ldx, cb, rows, out, ldo, s, parts);
}
