// bamd_prefill2.hip — the exact matrix-core prefill mat-mul with the A fragments BUILT ONCE PER WORKGROUP (Q4_K / Q5_K x Q8_K; up to 64 tokens Q6_K x Q8_K as well).
//
// Reference: ggml_compute_forward_mul_mat with ne11 = T (ggml.c:12277-12492) over ggml_vec_dot_q{4,5,6}_K_q8_K (ggml-quants.c:6832 / :7400 / :8037);
// the second implementation it is tested against is the integer-dot kernel of bamd_prefill.hip (matmul_batch_kernel): ONE
// v_mfma_f32_16x16x32_f16 per SIMD lane e of the reference gives the exact integer sums isum_e of a 16-row x 16-token tile, the f32 chains
// acc_e = fma(d_x d_y, isum_e, acc_e), the min terms and the final hsum tree follow on the VALU in the reference's order.
//
// Against kernels in which every wave builds its own fragments, and why: there every wave expands the nibbles of ITS 16 rows into f16 scale x quant
// fragments and uses each fragment for two MFMAs — 365 issued instructions per wave and super-block, ~150 of them that expansion and the header
// unpacking in front of it.  Here
//   * a workgroup is 64 rows x 64 tokens and every fragment is built ONCE per workgroup, one super-block AHEAD, into an LDS ring in MFMA operand layout
//     (ds_write_b128, read back with ds_read_b128), by builders that work in the wave-stream's own lane order (lane (r, e) of a record group holds the
//     halves of MFMA lanes (row, g = 0..3) of fragment e: one coalesced request per wave); the build of super-block ci + 1 is independent of the MFMAs of
//     ci and interleaved with them;
//   * everything the header unpacking produced per step is PRECOMPUTED AT LOAD TIME into a per-matrix side table ("prefill aux", 104 B per row and
//     super-block for Q4_K / Q5_K, 72 B for Q6_K: the MI355X has the HBM for it): the builders' per-(row, sub-block pair) scale operands
//     {s, -1024 s, s'/16, -64 s'} as packed f16 pairs, and the consumers' d, dmin as f32 plus the min-term MFMA operands {2 m_a, 2 m_b, m_a, m_b}, which
//     travel global -> LDS by DMA with the activation records;
//   * sixteen waves with one 16 x 16 tile each (matmul_mfma3_q4k_kernel: Q4_K / Q5_K), where the products of many tokens (bamd_prefill_wide.hip) would leave CUs idle;
//     up to 64 tokens, where 64-row blocks leave the chip idle, 16-row blocks of specialised waves (matmul_few_kernel).
// Same bits as those kernels (which are gone), a third fewer vector instructions per MFMA — and the same time: profiles/r06_prefill_ceiling.txt has
// what bounds it and the timing-only ceiling builds (-DBAMD_PREFILL_CEILING).
#include "bamd_device.h"
#include "bamd_mfma_common.h"
#include <type_traits>
#include <stdlib.h>

typedef _Float16 bamd_h2 __attribute__((ext_vector_type(2)));
union bamd_h2u { uint32_t u; bamd_h2 h; };

struct bamd_mma2_args {
    const uint8_t * w;               // wave-stream records of the matrix (bamd_formats.h)
    const uint8_t * ph;              // prefill aux, builder part:  [row block of 64][super-block]([e-half], Q6_K)[4 row tiles][64 MFMA lanes][16 B]
    const uint8_t * ch;              // prefill aux, consumer part: [row block of 64][super-block][4 row tiles][X_CH4_RT or X_CH6_RT B]
    float * out; const float * res;  // [T][ldo]
    const uint8_t * blob16;          // f16 activation records (quantize_batch_kernel)
    int K, T, nrows, nrows_pad, ldo;
    unsigned long long * dbg;        // -DX_TIMING builds: per-wave phase clocks of workgroup (0, 0) (tools/prefill_phase.py); else unused
};

// LDS map of the sixteen-wave kernel (byte offsets), each region twice
#define X_FR 1040                                          /* bytes between fragments: 1 KiB + 16 — the builder's 16-byte stores of eight lanes (one row, e = 0..7) then fall on eight
                                                              different bank quads (260 dwords = 4 mod 64); a fragment itself stays contiguous (lane * 16) for the consumers' ds_read_b128 */
#define X_AF_BYTES (32 * X_FR)                             /* A fragments of one super-block: 4 row tiles x 8 fragments */
#define X_BS_BYTES (64 * BAMD_B16_REC)                     /* 64 token records of one super-block (38 912 B) */
#define X_CH4_RT 640                                       /* Q4_K / Q5_K consumer header of a row tile: 16 x d f32 | 16 x dmin f32 | 16 x 4 x 8 B of min operands */
#define X_CH6_RT 64                                        /* Q6_K: 16 x d f32 */
#define X3_CHS 3072                                        /* Q4_K / Q5_K consumer headers of a row block and super-block in the side table: 4 x 640 B, padded to three DMA instructions */
#define X_AF0 0

// ---- load-time side tables ---------------------------------------------------------------------------------------------------
// grid (super-blocks, row tiles incl. the padding tiles of the last row block), 64 threads = the MFMA lanes (m = row of the tile, g)
template <bool Q5>
__global__ void __launch_bounds__(64) prefill_aux_q4k_kernel(const uint8_t * __restrict__ w, int nrows_pad, int nb, uint8_t * __restrict__ ph, uint8_t * __restrict__ ch) {
    constexpr uint32_t RECB = Q5 ? BAMD_RECB_Q5K : BAMD_RECB_Q4K, HDRO = Q5 ? 1280u : 1024u;
    const int ci = blockIdx.x, rtile = blockIdx.y, lane = threadIdx.x, m = lane & 15, g = lane >> 4;
    const int row = rtile * 16 + m;
    uint4 hd = { 0u, 0u, 0u, 0u };
    if (row < nrows_pad) hd = *(const uint4 *) (w + ((size_t) (row >> 3) * nb + ci) * RECB + HDRO + (row & 7) * 16);
    const uint32_t u0 = hd.y, u1 = hd.z, u2 = hd.w;                                               // ggml-quants.c:6928-6933
    const uint32_t sc03 = u0 & 0x3f3f3f3fu, mn03 = u1 & 0x3f3f3f3fu;
    const uint32_t sc47 = (u2 & 0x0f0f0f0fu) | (((u0 >> 6) & 0x03030303u) << 4);
    const uint32_t mn47 = ((u2 >> 4) & 0x0f0f0f0fu) | (((u1 >> 6) & 0x03030303u) << 4);
    // builder operands of lane (m, g): scales of sub-blocks 2g, 2g+1 of row m, every value an exact f16
    const uint32_t scw = ((g >> 1) ? sc47 : sc03) >> (16 * (g & 1));
    const _Float16 s_lo = (_Float16) (float) (scw & 0xffu), s_hi = (_Float16) (float) ((scw >> 8) & 0xffu);
    bamd_h2u o0, o1, o2, o3;
    o0.h = (bamd_h2) { s_lo, s_lo }; o1.h = (bamd_h2) { (_Float16) -1024.f * s_lo, (_Float16) -1024.f * s_lo };
    if (Q5) { o2.h = (bamd_h2) { s_hi, s_hi }; o3.h = (bamd_h2) { (_Float16) -1024.f * s_hi, (_Float16) -1024.f * s_hi }; }
    else    { o2.h = (bamd_h2) { (_Float16) 0.0625f * s_hi, (_Float16) 0.0625f * s_hi }; o3.h = (bamd_h2) { (_Float16) -64.f * s_hi, (_Float16) -64.f * s_hi }; }
    *(uint4 *) (ph + (((size_t) (rtile >> 2) * nb + ci) * 4 + (rtile & 3)) * 1024 + lane * 16) = (uint4) { o0.u, o1.u, o2.u, o3.u };
    uint8_t * c = ch + ((size_t) (rtile >> 2) * nb + ci) * X3_CHS + (rtile & 3) * X_CH4_RT;
    if (g == 0) { *(float *) (c + m * 4) = h2f(hd.x & 0xffffu); *(float *) (c + 64 + m * 4) = h2f(hd.x >> 16); }     // d of the 16 rows, then dmin of the 16 rows
    {   // min operands of pair l = g: {2 m_2l, 2 m_2l+1, m_2l, m_2l+1}
        const uint32_t mw = ((g >> 1) ? mn47 : mn03) >> (16 * (g & 1));
        const _Float16 ma = (_Float16) (float) (mw & 0xffu), mb = (_Float16) (float) ((mw >> 8) & 0xffu);
        bamd_h2u two, one; one.h = (bamd_h2) { ma, mb }; two.h = one.h + one.h;
        *(uint2 *) (c + 128 + m * 32 + g * 8) = (uint2) { two.u, one.u };
    }
}
// Q6_K: per lane (m, g) and e-half h the int8 scales of sub-blocks 2g, 2g+1 (record byte h*8 + c = file scales[2c + h]) split sc = sa + sl with
// sa = sc & ~15 (a multiple of 16 in [-128, 112]) and sl = sc & 15: sa x (q - 32) and sl x (q - 32) are exact f16 (|.| <= 4096 in steps of 16, <= 480)
__global__ void __launch_bounds__(64) prefill_aux_q6k_kernel(const uint8_t * __restrict__ w, int nrows_pad, int nb, uint8_t * __restrict__ ph, uint8_t * __restrict__ ch) {
    const int ci = blockIdx.x, rtile = blockIdx.y, lane = threadIdx.x, m = lane & 15, g = lane >> 4;
    const int row = rtile * 16 + m;
    uint4 sc = { 0u, 0u, 0u, 0u }; uint32_t d16 = 0u;
    if (row < nrows_pad) {
        const uint8_t * rec = w + ((size_t) (row >> 3) * nb + ci) * 1680;
        sc = *(const uint4 *) (rec + 1536 + (row & 7) * 16); d16 = *(const unsigned short *) (rec + 1664 + (row & 7) * 2);
    }
    const uint32_t scd[4] = { sc.x, sc.y, sc.z, sc.w };
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const uint32_t wv = scd[h * 2 + (g >> 1)] >> (16 * (g & 1));
        const int s0 = (int) (int8_t) (wv & 0xffu), s1 = (int) (int8_t) ((wv >> 8) & 0xffu);
        const _Float16 a0 = (_Float16) (float) (s0 & ~15), l0 = (_Float16) (float) (s0 & 15), a1 = (_Float16) (float) (s1 & ~15), l1 = (_Float16) (float) (s1 & 15);
        bamd_h2u o0, o1, o2, o3; o0.h = (bamd_h2) { a0, a0 }; o1.h = (bamd_h2) { l0, l0 }; o2.h = (bamd_h2) { a1, a1 }; o3.h = (bamd_h2) { l1, l1 };
        *(uint4 *) (ph + ((((size_t) (rtile >> 2) * nb + ci) * 2 + h) * 4 + (rtile & 3)) * 1024 + lane * 16) = (uint4) { o0.u, o1.u, o2.u, o3.u };
    }
    if (g == 0) *(float *) (ch + (((size_t) (rtile >> 2) * nb + ci) * 4 + (rtile & 3)) * X_CH6_RT + m * 4) = h2f(d16);
}

// ---- Q4_K / Q5_K: the sixteen-wave kernel further down (matmul_mfma3_q4k_kernel).  MFMA lane l = (m = l & 15, g = l >> 4): A row m, B token m, k-slots (g, i) =
//      (sub-block 2g + (i >> 2), u = i & 3); C/D rows 4g + i, token m.  (An eight-wave layout of the same arithmetic — 16 x 32 per wave, 96 accumulators, two waves
//      per SIMD — took 27.4 vs 25.4 ms per 512-token micro-batch, profiles/r06_prefill_ceiling.txt.)

// ==== sixteen waves ===========================================================================================================================
// Eight waves with two tiles each trade vector instructions for LDS traffic and gain nothing (two waves per SIMD: a step is a chain of dependent
// latencies).  This kernel puts four waves on every SIMD:
//   * a workgroup is SIXTEEN waves: four row tiles x four token tiles, ONE 16 x 16 tile per wave (48 accumulator registers, <= 118 VGPRs);
//     every A fragment is built once and read by four waves, every token record staged once and read by four;
//   * staging is three full-wave DMA instructions per wave and step, the same straight-line code on every wave: sources are fixed per-wave scalar pointers
//     plus per-lane offsets that advance by a per-wave stride (records 608 B, consumer headers 3 KiB, builder operands 4 KiB per super-block), destinations
//     per-wave constants; no clamping at the end of K (the last copies read one super-block past the tables — allocated with that slack — into a block
//     nobody reads again); the copies follow the MFMAs of e = 0..2 instead of opening the step (all sixteen waves' copies at once queue in the vector
//     memory path: every wave sat 500-1200 clocks in its issue stage);
//   * the builder's scale operands travel by DMA as well, two steps ahead, into the operand slot of the block that is being read (its previous content
//     was consumed one step earlier), so a wave's own loads are 8 bytes of nibbles per lane and step through a buffer descriptor (scalar offset);
//   * d_y sits inside the token record; the chain FMAs of e follow the MFMA of e + 2 (no MFMA -> VALU wait states); the epilogue stores 16 bytes per lane.
// 112 issued instructions per wave and step (one that builds its own fragments: 365 per two tiles).  What bounds it: profiles/r06_prefill_ceiling.txt.
#define X3_BLK (X_BS_BYTES + X3_CHS + 4096 + 32)           /* records (38 KiB) | headers (3 KiB) | operands (4 KiB) | 32 bytes of zeros: 46 112 B */
#define X3_BLK0 (2 * X_AF_BYTES)
#define X3_LDS_BYTES (X3_BLK0 + 2 * X3_BLK)                /* 158 784 B */
#define X3_CH_OFF X_BS_BYTES
#define X3_PH_OFF (X_BS_BYTES + X3_CHS)
#define X3_Z_OFF (X3_PH_OFF + 4096)
// one DMA instruction: 1 KiB from (scalar base + per-lane offset) to the LDS address lds_dst (m0 is saved and restored around it: the compiler reserves the register)
__device__ __forceinline__ void x3_dma(const void * sbase, uint32_t voff, uint32_t lds_dst) { lds_dma16_s(sbase, voff, lds_dst); }
#ifndef X_TIMING
#define X_TIMING 0
#endif
#ifndef BAMD_PREFILL_CEILING
#define BAMD_PREFILL_CEILING 0
#endif
#if X_TIMING
#define X_T(i_) do { const unsigned long long now_ = __builtin_readcyclecounter(); tacc[i_] += now_ - tlast; tlast = now_; } while (0)
#else
#define X_T(i_) do { } while (0)
#endif
template <int EPI, bool Q5>
__global__ void __launch_bounds__(1024) matmul_mfma3_q4k_kernel(bamd_mma2_args a) {
    constexpr uint32_t RECB = Q5 ? BAMD_RECB_Q5K : BAMD_RECB_Q4K;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const int tid = threadIdx.x, lane = tid & 63, wave = wave_id(), m = lane & 15, g = lane >> 4;
    const int rt = wave >> 2, tt = wave & 3;
    const int nb = a.K >> 8;
    const int rb = blockIdx.y, t0 = blockIdx.x * 64;
    const int rtg = rb * 4 + rt;
    const bool live = rtg * 16 < a.nrows_pad;
    const uint32_t rstep = BAMD_B16_STEP(a.T);             // records of a super-block: all tokens' one behind the other
    const uint32_t lds0 = (uint32_t) (size_t) (bamd_lds_vp) smem;
    // ---- stage plan.  A block = 45 KiB-instructions: k = 0..37 records (chunk 64 k + lane of 64 tokens x 38), 38..40 consumer headers, 41..44 builder
    //      operands.  Wave w issues k = w, 16 + w and k2 = 32 + w (w <= 12; waves 13..15 repeat the operand copies 41..43: same bytes, same place).
    auto rec_off = [&](int idx) { const int tok = idx / BAMD_B16_Q, q = idx - tok * BAMD_B16_Q; const int tg = t0 + tok < a.T ? t0 + tok : a.T - 1; return (uint32_t) tg * BAMD_B16_MEM + (uint32_t) q * 16u; };
    const int k2 = wave <= 12 ? 32 + wave : 28 + wave;
    const bool rec2 = k2 <= 37, hdr2 = k2 >= 38 && k2 <= 40;
    uint32_t so0 = rec_off(tid), so1 = rec_off(1024 + tid);          // advance by one super-block per step (sources stay fixed scalar pointers)
    uint32_t so2 = rec2 ? rec_off(k2 * 64 + lane) : (uint32_t) (((hdr2 ? k2 - 38 : k2 - 41) * 64 + lane) * 16);
    // sources of the NEXT stage call (the first call stages super-block 0 and the operands of super-block 1)
    const uint8_t * p01 = a.blob16;
    const uint8_t * p2 = rec2 ? a.blob16 : hdr2 ? a.ch + (size_t) rb * nb * X3_CHS : a.ph + (size_t) rb * nb * 4096 + 4096;
    const uint32_t st2 = rec2 ? rstep : hdr2 ? (uint32_t) X3_CHS : 4096u;
    // destinations by the parity of the step that issues the copies: records / headers of ci + 1 -> the OTHER block, operands of ci + 2 -> the block in use
    const uint32_t blk_a = lds0 + X3_BLK0, blk_b = blk_a + X3_BLK;
    const uint32_t d0_even = blk_b + (uint32_t) wave * 1024u, d0_odd = blk_a + (uint32_t) wave * 1024u;
    const uint32_t d2_even = (k2 <= 40 ? blk_b : blk_a) + (uint32_t) k2 * 1024u, d2_odd = (k2 <= 40 ? blk_a : blk_b) + (uint32_t) k2 * 1024u;
#define X3_STAGE(PAR) do { x3_dma(p01, so0, (PAR) ? d0_odd : d0_even); x3_dma(p01, so1, ((PAR) ? d0_odd : d0_even) + 16384u); x3_dma(p2, so2, (PAR) ? d2_odd : d2_even); \
                           so0 += rstep; so1 += rstep; so2 += st2; } while (0)
    // ---- builder: wave (rt, tt) = record group q = tt & 1 of the row tile, pieces g = 2 gh + j (gh = tt >> 1, j = 0, 1): lane (r, e) holds dwords 2 gh, 2 gh + 1
    //      of stream lane (r, e) = the halves of MFMA lanes (8 q + r, 2 gh + j) of fragment e
    const int br = lane >> 3, be = lane & 7, bq = tt & 1, gh = tt >> 1;
    const int rgq = 2 * (live ? rtg : rb * 4) + bq;
    const int rgc = rgq * 8 < a.nrows_pad ? rgq : rgq - 1;            // a last tile of 8 (padded) rows: its first record group twice (rows 8..15 are never stored)
    const __amdgpu_buffer_rsrc_t wrs = __builtin_amdgcn_make_buffer_rsrc((void *) uniform_ptr(a.w + (size_t) rgc * nb * RECB), 0, 0x7fffffff, 0x00020000);
    const int vraw = lane * 16 + gh * 8, vqh = 1024 + lane * 4;
    uint2 raw[2]; uint32_t qh[2];
    auto load_set = [&](int ci, auto set_tag) {
        constexpr int S = decltype(set_tag)::value;
        const u32x2_t v = __builtin_amdgcn_raw_buffer_load_b64(wrs, vraw, ci * (int) RECB, 0); raw[S] = make_uint2(v.x, v.y);
        if (Q5) qh[S] = __builtin_amdgcn_raw_buffer_load_b32(wrs, vqh, ci * (int) RECB, 0);
    };
    bamd_h2u c0, c1, c2, c3;
    const uint32_t qs0 = 4u * (uint32_t) gh;
    auto build_a = [&](uint32_t wq, uint32_t q, int j) {
        uint32_t lo = wq & 0x0f0f0f0fu, hi = Q5 ? (wq >> 4) & 0x0f0f0f0fu : wq & 0xf0f0f0f0u;      // Q4_K: the high nibbles stay in place (16 n; the scale operand is s / 16)
        if (Q5) { lo |= ((q >> (qs0 + 2 * j)) & 0x01010101u) << 4; hi |= ((q >> (qs0 + 2 * j + 1)) & 0x01010101u) << 4; }
        c0.u = __builtin_amdgcn_perm(0x64646464u, lo, 0x04010400u); c1.u = __builtin_amdgcn_perm(0x64646464u, lo, 0x04030402u);
        c2.u = __builtin_amdgcn_perm(0x64646464u, hi, 0x04010400u); c3.u = __builtin_amdgcn_perm(0x64646464u, hi, 0x04030402u);
    };
    auto build_b = [&](const uint4 & s, unsigned char * dst) {
        bamd_h2u s0, n0, s1, n1, a0, a1, a2, a3; s0.u = s.x; n0.u = s.y; s1.u = s.z; n1.u = s.w;
        a0.h = __builtin_elementwise_fma(c0.h, s0.h, n0.h); a1.h = __builtin_elementwise_fma(c1.h, s0.h, n0.h);     // (1024 + n) s - 1024 s = n s, one rounding, exact
        a2.h = __builtin_elementwise_fma(c2.h, s1.h, n1.h); a3.h = __builtin_elementwise_fma(c3.h, s1.h, n1.h);
        *(uint4 *) dst = (uint4) { a0.u, a1.u, a2.u, a3.u };
    };
    // per-lane LDS addresses (first copy of each region)
    unsigned char * afw = smem + X_AF0 + (rt * 8 + be) * X_FR + ((2 * gh) * 16 + 8 * bq + br) * 16;
    const unsigned char * afr = smem + X_AF0 + rt * 8 * X_FR + lane * 16;
    const unsigned char * phl = smem + X3_BLK0 + X3_PH_OFF + rt * 1024 + (2 * gh) * 256 + (8 * bq + br) * 16;
    const unsigned char * tok = smem + X3_BLK0 + (size_t) (tt * 16 + m) * BAMD_B16_REC;                  // this lane's token record
    const unsigned char * bop = tok + g * 16;
    const unsigned char * bmn = tok + 512 + (Q5 ? g * 8 : 0);
    const unsigned char * chd = smem + X3_BLK0 + X3_CH_OFF + rt * X_CH4_RT + g * 16;                // d of rows 4g .. 4g+3; their dmin 64 bytes on
    const unsigned char * cmn = Q5 ? smem + X3_BLK0 + X3_CH_OFF + rt * X_CH4_RT + 128 + m * 32 + g * 8
                                   : (g == 0 ? smem + X3_BLK0 + X3_CH_OFF + rt * X_CH4_RT + 128 + m * 32 : smem + X3_BLK0 + X3_Z_OFF);
    bamd_f4 acc[8], accm[4];
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e] = (bamd_f4) { 0.f, 0.f, 0.f, 0.f };
#pragma unroll
    for (int l = 0; l < 4; ++l) accm[l] = (bamd_f4) { 0.f, 0.f, 0.f, 0.f };
    // prologue = the staging half of a step "-1" of odd parity: records / headers of super-block 0 into block a, operands of super-block 1 into block b;
    // the fragments of super-block 0 are built with operands straight from memory
    if (tid < 16) *(uint32_t *) (smem + X3_BLK0 + X3_Z_OFF + (tid >> 3) * X3_BLK + (tid & 7) * 4) = 0u;
    X3_STAGE(1);
    load_set(0, std::integral_constant<int, 0>());
    load_set(1, std::integral_constant<int, 1>());               // (no clamping at the end of K: the wave-stream copies are allocated with 4 KiB of slack, bamd_engine.cpp dev_alloc)
    {
        const uint8_t * p0 = a.ph + (size_t) rb * nb * 4096 + (size_t) rt * 1024 + (size_t) ((2 * gh) * 256 + (8 * bq + br) * 16);
        const uint4 s0 = *(const uint4 *) p0, s1 = *(const uint4 *) (p0 + 256);
        build_a(raw[0].x, Q5 ? qh[0] : 0u, 0); build_b(s0, afw);
        build_a(raw[0].y, Q5 ? qh[0] : 0u, 1); build_b(s1, afw + 256);
    }
    lds_dma_wait();
    __syncthreads();
#if X_TIMING
    unsigned long long tacc[8] = { 0, 0, 0, 0, 0, 0, 0, 0 }, tlast = __builtin_readcyclecounter();
#endif
    auto step = [&](const int ci, auto cur_tag) {
        constexpr int CUR = decltype(cur_tag)::value, NXT = CUR ^ 1;
        X_T(0);
        float D[4], Dm[4];
        const bamd_f4 h0 = *(const bamd_f4 *) (chd + CUR * X3_BLK), h1 = *(const bamd_f4 *) (chd + CUR * X3_BLK + 64);
        const float ydv = *(const float *) (tok + CUR * X3_BLK + 560);
        D[0] = ydv * h0[0]; D[1] = ydv * h0[1]; D[2] = ydv * h0[2]; D[3] = ydv * h0[3];
        Dm[0] = (-ydv) * h1[0]; Dm[1] = (-ydv) * h1[1]; Dm[2] = (-ydv) * h1[2]; Dm[3] = (-ydv) * h1[3];
        {
            // The step opens with operand reads and MFMAs; the three staging copies and the nibble load of this wave follow the MFMAs of e = 0..3 one by
            // one (issued together at the top they queue behind the other fifteen waves' copies — the vector memory path takes 64 B per clock — and every
            // wave sits in its issue stage for 500-1200 clocks before its first MFMA: tools/prefill_phase.py); the fragment pieces of the next
            // super-block are built beside e = 4..7
            // the chain FMAs of e follow the MFMA of e + 2 (one iteration behind, the compiler pads every MFMA -> VALU read with s_nop 1..6: ten issue slots per step)
            bamd_h8 Aq[3], Bq[3]; bamd_f4 sp[2];
#if BAMD_PREFILL_CEILING
            bamd_f4 csum = { 0.f, 0.f, 0.f, 0.f }, csum2 = { 0.f, 0.f, 0.f, 0.f };
            const unsigned char * afr2 = smem + X_AF0 + (rt ^ 1) * 8 * X_FR + lane * 16;
            (void) afr2; (void) csum2;
#endif
#define X_LDA(e_) (*(const bamd_h8 *) (afr + CUR * X_AF_BYTES + (e_) * X_FR))
#define X_LDB(e_) (*(const bamd_h8 *) (bop + CUR * X3_BLK + (e_) * 64))
            Aq[0] = X_LDA(0); Bq[0] = X_LDB(0); Aq[1] = X_LDA(1); Bq[1] = X_LDB(1);
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                if (e + 2 < 8) { Aq[(e + 2) % 3] = X_LDA(e + 2); Bq[(e + 2) % 3] = X_LDB(e + 2); }
                if (e >= 4 && (e & 1) == 0) build_a(e == 4 ? raw[NXT].x : raw[NXT].y, Q5 ? qh[NXT] : 0u, (e >> 1) & 1);
                const bamd_f4 z = { 0.f, 0.f, 0.f, 0.f };
#if BAMD_PREFILL_CEILING
                // TIMING-ONLY ceiling builds (tools/prefill_ceiling.sh; never shipped, results are garbage): what the exact arithmetic's EIGHT separate per-lane sums per
                // super-block cost.  1: the eight MFMAs of a step accumulate into ONE accumulator (K = 256) and ONE chain FMA per super-block and tile follows — same
                // operand traffic, same staging, same fragment build.  2: the same, and every B operand read serves the MFMAs of TWO row tiles (this wave's and its
                // neighbour's A fragments: 1.5 KB of LDS reads per MFMA instead of 2; the launcher halves the row blocks so that the MFMA count stays what it was)
                csum = __builtin_amdgcn_mfma_f32_16x16x32_f16(Aq[e % 3], Bq[e % 3], e == 0 ? z : csum, 0, 0, 0);
                if (BAMD_PREFILL_CEILING == 2) csum2 = __builtin_amdgcn_mfma_f32_16x16x32_f16(*(const bamd_h8 *) (afr2 + CUR * X_AF_BYTES + e * X_FR), Bq[e % 3], e == 0 ? z : csum2, 0, 0, 0);
                const bamd_f4 si = z;
#else
                const bamd_f4 si = __builtin_amdgcn_mfma_f32_16x16x32_f16(Aq[e % 3], Bq[e % 3], z, 0, 0, 0);
#endif
                if (e == 0) x3_dma(p01, so0, CUR ? d0_odd : d0_even);
                if (e == 1) x3_dma(p01, so1, (CUR ? d0_odd : d0_even) + 16384u);
                if (e == 2) { x3_dma(p2, so2, CUR ? d2_odd : d2_even); so0 += rstep; so1 += rstep; so2 += st2; }
                if (e == 3) load_set(ci + 2, std::integral_constant<int, CUR>());
#if !BAMD_PREFILL_CEILING
                if (e > 1) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) acc[e - 2][i] = fmaf(D[i], sp[e & 1][i], acc[e - 2][i]);
                }
#endif
                if (e >= 4 && (e & 1)) build_b(*(const uint4 *) (phl + NXT * X3_BLK + ((e >> 1) & 1) * 256), afw + NXT * X_AF_BYTES + ((e >> 1) & 1) * 256);
                sp[e & 1] = si;
                __builtin_amdgcn_sched_barrier(0);
                if (e == 3) X_T(1);
            }
#if BAMD_PREFILL_CEILING
#pragma unroll
            for (int i = 0; i < 4; ++i) { acc[0][i] = fmaf(D[i], csum[i], acc[0][i]); if (BAMD_PREFILL_CEILING == 2) acc[1][i] = fmaf(D[i], csum2[i], acc[1][i]); }
            (void) sp;
#else
#pragma unroll
            for (int i = 0; i < 4; ++i) { acc[6][i] = fmaf(D[i], sp[0][i], acc[6][i]); acc[7][i] = fmaf(D[i], sp[1][i], acc[7][i]); }
#endif
#undef X_LDA
#undef X_LDB
        }
        X_T(2);
        if (Q5) {
            union { uint2 u; bamd_h4 h; } av, bv; av.u = *(const uint2 *) (cmn + CUR * X3_BLK); bv.u = *(const uint2 *) (bmn + CUR * X3_BLK);
            const bamd_f4 z = { 0.f, 0.f, 0.f, 0.f };
            const bamd_f4 pm = __builtin_amdgcn_mfma_f32_16x16x16f16(av.h, bv.h, z, 0, 0, 0);
#pragma unroll
            for (int i = 0; i < 4; ++i) { const float t = Dm[i] * pm[i]; accm[0][i] = accm[0][i] + t; }
        } else {
            const uint4 ma = *(const uint4 *) (cmn + CUR * X3_BLK), mb = *(const uint4 *) (cmn + CUR * X3_BLK + 16);
            const uint4 sfa = *(const uint4 *) (bmn + CUR * X3_BLK), sfb = *(const uint4 *) (bmn + CUR * X3_BLK + 16);
            const uint2 al[4] = { { ma.x, ma.y }, { ma.z, ma.w }, { mb.x, mb.y }, { mb.z, mb.w } };
            const uint2 bl[4] = { { sfa.x, sfa.y }, { sfa.z, sfa.w }, { sfb.x, sfb.y }, { sfb.z, sfb.w } };
            bamd_f4 pm[4];
#pragma unroll
            for (int l = 0; l < 4; ++l) {
                union { uint2 u; bamd_h4 h; } av4, bv4; av4.u = al[l]; bv4.u = bl[l];
                const bamd_f4 z = { 0.f, 0.f, 0.f, 0.f };
                pm[l] = __builtin_amdgcn_mfma_f32_16x16x16f16(av4.h, bv4.h, z, 0, 0, 0);
            }
#pragma unroll
            for (int l = 0; l < 4; ++l) {
#pragma unroll
                for (int i = 0; i < 4; ++i) accm[l][i] = fmaf(Dm[i], pm[l][i], accm[l][i]);
            }
        }
        X_T(3);
        lds_dma_wait();
        X_T(4);
        __syncthreads();
        X_T(5);
    };
    for (int ci = 0; ci < nb; ci += 2) {
        step(ci, std::integral_constant<int, 0>());
        if (ci + 1 < nb) step(ci + 1, std::integral_constant<int, 1>());
    }
#undef X3_STAGE
#if X_TIMING
    if (a.dbg && blockIdx.x == 0 && blockIdx.y == (gridDim.y >> 1) && lane == 0) {
#pragma unroll
        for (int i = 0; i < 6; ++i) a.dbg[wave * 8 + i] = tacc[i];
        a.dbg[wave * 8 + 6] = (unsigned long long) nb;
    }
#endif
    if (!live) return;
    // hsum_float_8 over e and the acc_m folds, in the reference's order (finish_row), then the epilogue: rows 4g .. 4g+3 of token t are 16 consecutive bytes
    const int t = t0 + tt * 16 + m;
    float val[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float v = ((acc[0][i] + acc[4][i]) + (acc[2][i] + acc[6][i])) + ((acc[1][i] + acc[5][i]) + (acc[3][i] + acc[7][i]));
        const float mm = Q5 ? accm[0][i] : (accm[0][i] + accm[2][i]) + (accm[1][i] + accm[3][i]);
        val[i] = v + mm;
    }
    const int row0 = rtg * 16 + 4 * g;
    if (t < a.T && row0 < a.nrows) {
        const size_t o = (size_t) t * a.ldo + row0;
        if (row0 + 3 < a.nrows && (a.ldo & 3) == 0) {
            bamd_f4 y = { val[0], val[1], val[2], val[3] };
            if (EPI != BAMD_EPI_STORE) {
                const bamd_f4 r = *(const bamd_f4 *) (a.res + o);
#pragma unroll
                for (int i = 0; i < 4; ++i) y[i] = EPI == BAMD_EPI_ADD ? val[i] + r[i] : v_silu(r[i]) * val[i];
            }
            *(bamd_f4 *) (a.out + o) = y;
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (row0 + i < a.nrows) a.out[o + i] = EPI == BAMD_EPI_ADD ? val[i] + a.res[o + i] : EPI == BAMD_EPI_SILU_MUL ? v_silu(a.res[o + i]) * val[i] : val[i];
        }
    }
}

// ==== few tokens ==============================================================================================================================
// A prompt of up to 64 tokens leaves the kernels above without work for the chip: 64-row blocks make 64 of them at 4096 rows, and each walks all of K behind a barrier per
// super-block that waits for everything it has requested (1.5 us per super-block: 25 us at K = 4096, 77 and, Q6_K, 105 us at K = 14336, whatever the tokens).  Here a block is ONE
// row tile (16 rows) x up to 16 NTT tokens on twelve waves, one of each kind per SIMD: wave tt < 4 takes token tile tt, four build a quarter of the next super-block's fragments
// each, four copy (all of it one after the other on four waves: 1230 ns a super-block at 37 tokens; copies spread over consumers and builders: 930 — a copy holds its wave until
// the vector memory path takes it); the arithmetic, its order and the layouts are those above.  Everything a step reads travels global -> LDS by DMA — token records two
// super-blocks ahead, the row tile's quants, scales and headers four — and the wait at the end of a step leaves what was issued in it (and the weights issued in the one before)
// in flight, so that a step is not as long as the memory's latency.  37 tokens, 4096 rows, launches one behind the other, 64-row blocks and this: K = 4096 24.7 and 11.3 us, K = 14336 77
// and 31.4 (Q5_K 74 and 32.1, Q6_K on matmul_wide_kernel 84 and 44.6).  The copies of the token records are the same to every block: of the tokens that there are and half a line out of step
// (BAMD_B16_MEM), a launch in a prompt 38 -> 34.6 us, a prompt 4681 -> 4511 (48 tokens, no fewer copies, level).  Without them the 31.4 us are 27.4 (Q6_K 38.5 of 44.6, 48 tokens 27.5 of 34.4).
//   W slot of a super-block   Q4_K / Q5_K: 2 x 1 KiB quants of the two record groups | 1 KiB builder operands | 1 KiB consumer header | Q5_K: 2 x 256 B fifth bits
//                             Q6_K: 2 x 1 KiB low bits | 2 x 512 B high bits | 2 x 1 KiB builder operands of the e-halves | 64 B of d
template <int TYPE> struct FewW { static constexpr int SLOT = TYPE == BAMD_Q6_K ? 5184 : TYPE == BAMD_Q5_K ? 4608 : 4096, COPIES = TYPE == BAMD_Q4_K ? 1 : 2; };
#define XF_RING 3                                         /* super-blocks of token records in LDS */
#define XF_WRING 5                                        /* of the row tile's operands */
constexpr int few_records(int ntt) { return (ntt * 16 * BAMD_B16_Q + 63) / 64; }       /* KiB of token records of a super-block */
constexpr size_t few_lds(int type, int ntt) {
    return (size_t) 16 * X_FR + (size_t) XF_RING * few_records(ntt) * 1024 + (size_t) XF_WRING * (type == BAMD_Q6_K ? FewW<BAMD_Q6_K>::SLOT : type == BAMD_Q5_K ? FewW<BAMD_Q5_K>::SLOT : FewW<BAMD_Q4_K>::SLOT) + 32;
}
template <int TYPE, int EPI, int NTT>
__device__ __forceinline__ void few_block(const bamd_mma2_args & a, int rtg) {
    constexpr bool Q5 = TYPE == BAMD_Q5_K, Q6 = TYPE == BAMD_Q6_K;
    constexpr uint32_t RECB = Q6 ? 1680u : Q5 ? BAMD_RECB_Q5K : BAMD_RECB_Q4K;
    constexpr int RS = few_records(NTT) * 1024, NW = FewW<TYPE>::COPIES, WS = FewW<TYPE>::SLOT;
    constexpr int REC0 = 16 * X_FR, W0 = REC0 + XF_RING * RS, Z0 = W0 + XF_WRING * WS;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const int tid = threadIdx.x, lane = tid & 63, wave = wave_id(), tt = wave, bw = wave & 3, m = lane & 15, g = lane >> 4;
    const int nb = a.K >> 8, rb = rtg >> 2, rtl = rtg & 3, t0 = blockIdx.x * (16 * NTT);
    const uint32_t lds0 = (uint32_t) (size_t) (bamd_lds_vp) smem;
    const bool active = tt < NTT && t0 + tt * 16 < a.T, builder = (wave >> 2) == 1, copier = wave >= 8;
    // the row tile's operands: a kilobyte per copier, and the fifth bits / high bits and d of Q5_K / Q6_K.  A last tile of 8 (padded) rows takes its first record group twice
    // (rows 8..15 are never stored)
    const int rgq = 2 * rtg + (bw & 1), rgc = rgq * 8 < a.nrows_pad ? rgq : rgq - 1;
    const uint8_t * rec = a.w + (size_t) rgc * nb * RECB, * s1, * s2; uint32_t st1, st2, d1, d2; int n2;
    if (bw < 2) { s1 = rec; st1 = RECB; d1 = (uint32_t) bw * 1024u; s2 = rec + 1024; st2 = RECB; d2 = Q6 ? 2048u + bw * 512u : 4096u + bw * 256u; n2 = Q6 ? 32 : 16; }
    else {
        if (Q6) { s1 = a.ph + ((size_t) rb * nb * 2 + (bw & 1)) * 4096 + (size_t) rtl * 1024; st1 = 8192u; d1 = 3072u + (bw & 1) * 1024u; }
        else if (bw == 2) { s1 = a.ph + (size_t) rb * nb * 4096 + (size_t) rtl * 1024; st1 = 4096u; d1 = 2048u; }
        else { s1 = a.ch + (size_t) rb * nb * X3_CHS + (size_t) rtl * X_CH4_RT; st1 = X3_CHS; d1 = 3072u; }       // (640 B are used; a kilobyte from the last row tile ends inside the 3 KiB)
        s2 = s1; st2 = st1; d2 = d1; n2 = 1;                      // (every copier issues the same number of instructions: this one copies its first bytes again)
        if (Q6 && bw == 2) { s2 = a.ch + ((size_t) rb * nb * 4 + rtl) * X_CH6_RT; st2 = 4 * X_CH6_RT; d2 = 5120u; n2 = 4; }
    }
    auto copy_weights = [&](int ci, int slot) {
        const size_t k = (size_t) (ci < nb ? ci : nb - 1);
        const uint32_t w = lds0 + W0 + (uint32_t) slot * WS;
        const void * p1 = uniform_ptr(s1 + k * st1), * p2 = uniform_ptr(s2 + k * st2);
        lds_dma16_s(p1, (uint32_t) lane * 16u, w + d1);
        if (NW == 2 && lane < n2) lds_dma16_s(p2, (uint32_t) lane * 16u, w + d2);
    };
    // ---- builder: Q4_K / Q5_K as in the sixteen-wave kernel (record group bq, pieces 2 gh, 2 gh + 1); Q6_K: record group bq, piece gh of both pairs
    const int bq = bw & 1, gh = bw >> 1, br = Q6 ? (lane >> 2) & 7 : lane >> 3, be = Q6 ? lane & 3 : lane & 7, bp = lane >> 5;
    auto build45 = [&](const unsigned char * w, unsigned char * fr) {
        const uint2 raw = *(const uint2 *) (w + bq * 1024 + lane * 16 + gh * 8);
        const uint32_t q = Q5 ? *(const uint32_t *) (w + 4096 + bq * 256 + lane * 4) : 0u, qs0 = 4u * (uint32_t) gh;
        const unsigned char * p = w + 2048 + (2 * gh) * 256 + (8 * bq + br) * 16;
        unsigned char * dst = fr + be * X_FR + ((2 * gh) * 16 + 8 * bq + br) * 16;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const uint32_t wq = j ? raw.y : raw.x;
            const uint4 s = *(const uint4 *) (p + j * 256);
            uint32_t lo = wq & 0x0f0f0f0fu, hi = Q5 ? (wq >> 4) & 0x0f0f0f0fu : wq & 0xf0f0f0f0u;      // Q4_K: the high nibbles stay in place (16 n; the scale operand is s / 16)
            if (Q5) { lo |= ((q >> (qs0 + 2 * j)) & 0x01010101u) << 4; hi |= ((q >> (qs0 + 2 * j + 1)) & 0x01010101u) << 4; }
            bamd_h2u c0, c1, c2, c3, s0, n0, s1h, n1, a0, a1, a2, a3; s0.u = s.x; n0.u = s.y; s1h.u = s.z; n1.u = s.w;
            c0.u = __builtin_amdgcn_perm(0x64646464u, lo, 0x04010400u); c1.u = __builtin_amdgcn_perm(0x64646464u, lo, 0x04030402u);
            c2.u = __builtin_amdgcn_perm(0x64646464u, hi, 0x04010400u); c3.u = __builtin_amdgcn_perm(0x64646464u, hi, 0x04030402u);
            a0.h = __builtin_elementwise_fma(c0.h, s0.h, n0.h); a1.h = __builtin_elementwise_fma(c1.h, s0.h, n0.h);     // (1024 + n) s - 1024 s = n s, one rounding, exact
            a2.h = __builtin_elementwise_fma(c2.h, s1h.h, n1.h); a3.h = __builtin_elementwise_fma(c3.h, s1h.h, n1.h);
            *(uint4 *) (dst + j * 256) = (uint4) { a0.u, a1.u, a2.u, a3.u };
        }
    };
    auto build6 = [&](const unsigned char * w, int h, unsigned char * fr) {
        const uint2 q = *(const uint2 *) (w + bq * 1024 + (br * 8 + be) * 16 + bp * 8 + h * 64);
        const uint32_t hq = *(const uint32_t *) (w + 2048 + bq * 512 + (br * 8 + be) * 8 + bp * 4 + h * 32), sh = 4u * (uint32_t) gh;
        const uint4 s = *(const uint4 *) (w + 3072 + h * 1024 + (2 * bp + gh) * 256 + (8 * bq + br) * 16);
        const bamd_h2 k1056 = { (_Float16) -1056.f, (_Float16) -1056.f };
        const uint32_t uA = (__builtin_amdgcn_alignbit(hq, hq, (28u + sh) & 31u) & 0x30303030u) | ((q.x >> sh) & 0x0f0f0f0fu);
        const uint32_t uB = (__builtin_amdgcn_alignbit(hq, hq, (30u + sh) & 31u) & 0x30303030u) | ((q.y >> sh) & 0x0f0f0f0fu);
        bamd_h2u c, sa0, sl0, sa1, sl1, x0, x1, x2, x3; sa0.u = s.x; sl0.u = s.y; sa1.u = s.z; sl1.u = s.w;
        bamd_h2 v0, v1, v2, v3;
        c.u = __builtin_amdgcn_perm(0x64646464u, uA, 0x04010400u); v0 = c.h + k1056;      // (1024 + q) - 1056 = q - 32, exact
        c.u = __builtin_amdgcn_perm(0x64646464u, uA, 0x04030402u); v1 = c.h + k1056;
        c.u = __builtin_amdgcn_perm(0x64646464u, uB, 0x04010400u); v2 = c.h + k1056;
        c.u = __builtin_amdgcn_perm(0x64646464u, uB, 0x04030402u); v3 = c.h + k1056;
        unsigned char * dst = fr + be * (2 * X_FR) + ((2 * bp + gh) * 16 + 8 * bq + br) * 16;
        x0.h = v0 * sa0.h; x1.h = v1 * sa0.h; x2.h = v2 * sa1.h; x3.h = v3 * sa1.h;
        *(uint4 *) dst = (uint4) { x0.u, x1.u, x2.u, x3.u };
        x0.h = v0 * sl0.h; x1.h = v1 * sl0.h; x2.h = v2 * sl1.h; x3.h = v3 * sl1.h;
        *(uint4 *) (dst + X_FR) = (uint4) { x0.u, x1.u, x2.u, x3.u };
    };
    unsigned char * const fr0 = smem, * const fr1 = smem + 8 * X_FR;
    bamd_f4 acc[8], accm[4];
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e] = (bamd_f4) { 0.f, 0.f, 0.f, 0.f };
#pragma unroll
    for (int l = 0; l < 4; ++l) accm[l] = (bamd_f4) { 0.f, 0.f, 0.f, 0.f };
    const bamd_f4 z = { 0.f, 0.f, 0.f, 0.f };
    const unsigned char * const zero = smem + Z0;
    auto consume45 = [&](const unsigned char * recs, const unsigned char * w, const unsigned char * fr) {
        const unsigned char * tok = recs + (size_t) (tt * 16 + m) * BAMD_B16_REC, * ch = w + 3072;
        // every operand of the super-block is requested before the first matrix instruction (left to itself the compiler reads two, waits, multiplies: eight LDS latencies in a row)
        bamd_h8 A[8], B[8]; uint4 ma, mb, sfa, sfb; uint2 m5, s5;
#pragma unroll
        for (int e = 0; e < 8; ++e) { A[e] = *(const bamd_h8 *) (fr + e * X_FR + lane * 16); B[e] = *(const bamd_h8 *) (tok + g * 16 + e * 64); }
        const bamd_f4 h0 = *(const bamd_f4 *) (ch + g * 16), h1 = *(const bamd_f4 *) (ch + 64 + g * 16);
        const float ydv = *(const float *) (tok + 560);
        if constexpr (Q5) { m5 = *(const uint2 *) (ch + 128 + m * 32 + g * 8); s5 = *(const uint2 *) (tok + 512 + g * 8); }
        else {
            const unsigned char * cm = g == 0 ? ch + 128 + m * 32 : zero;
            ma = *(const uint4 *) cm; mb = *(const uint4 *) (cm + 16); sfa = *(const uint4 *) (tok + 512); sfb = *(const uint4 *) (tok + 528);
        }
        __builtin_amdgcn_sched_barrier(0);
        bamd_f4 si[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) si[e] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A[e], B[e], z, 0, 0, 0);
        float D[4], Dm[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) { D[i] = ydv * h0[i]; Dm[i] = (-ydv) * h1[i]; }
#pragma unroll
        for (int e = 0; e < 8; ++e)
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[e][i] = fmaf(D[i], si[e][i], acc[e][i]);
        if constexpr (Q5) {
            union { uint2 u; bamd_h4 h; } av, bv; av.u = m5; bv.u = s5;
            const bamd_f4 pm = __builtin_amdgcn_mfma_f32_16x16x16f16(av.h, bv.h, z, 0, 0, 0);
#pragma unroll
            for (int i = 0; i < 4; ++i) { const float t = Dm[i] * pm[i]; accm[0][i] = accm[0][i] + t; }
        } else {
            const uint2 al[4] = { { ma.x, ma.y }, { ma.z, ma.w }, { mb.x, mb.y }, { mb.z, mb.w } };
            const uint2 bl[4] = { { sfa.x, sfa.y }, { sfa.z, sfa.w }, { sfb.x, sfb.y }, { sfb.z, sfb.w } };
            bamd_f4 pm[4];
#pragma unroll
            for (int l = 0; l < 4; ++l) { union { uint2 u; bamd_h4 h; } av, bv; av.u = al[l]; bv.u = bl[l]; pm[l] = __builtin_amdgcn_mfma_f32_16x16x16f16(av.h, bv.h, z, 0, 0, 0); }
#pragma unroll
            for (int l = 0; l < 4; ++l)
#pragma unroll
                for (int i = 0; i < 4; ++i) accm[l][i] = fmaf(Dm[i], pm[l][i], accm[l][i]);
        }
    };
    auto consume6 = [&](const unsigned char * recs, const unsigned char * w, const unsigned char * fr, auto h_tag) {
        constexpr int H = decltype(h_tag)::value;
        const unsigned char * tok = recs + (size_t) (tt * 16 + m) * BAMD_B16_REC;
        const bamd_f4 dw = *(const bamd_f4 *) (w + 5120 + g * 16);
        const float ydv = *(const float *) (tok + 560);
        float D[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) D[i] = ydv * dw[i];
        bamd_f4 s[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {                             // (requested all at once, as above, they hold up the builders, who set the pace here: 52 instead of 46 us)
            const bamd_h8 b = *(const bamd_h8 *) (tok + g * 16 + (4 * H + e) * 64);
            const bamd_f4 hi = __builtin_amdgcn_mfma_f32_16x16x32_f16(*(const bamd_h8 *) (fr + e * (2 * X_FR) + lane * 16), b, z, 0, 0, 0);
            s[e] = __builtin_amdgcn_mfma_f32_16x16x32_f16(*(const bamd_h8 *) (fr + e * (2 * X_FR) + X_FR + lane * 16), b, hi, 0, 0, 0);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[4 * H + e][i] = fmaf(D[i], s[e][i], acc[4 * H + e][i]);
    };
    auto barrier = [&] { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); __builtin_amdgcn_s_barrier(); asm volatile("" ::: "memory"); };
    if (tid < 8) *(uint32_t *) (smem + Z0 + tid * 4) = 0u;
    // a loop per kind of wave, barrier for barrier alike (one loop with branches inside moves the 48 accumulators through every join)
    auto after = [](int s, int by, int ring) { s += by; return s < ring ? s : s - ring; };
    if (copier) {
        // Token records lie one token behind the other (quantize_batch_kernel): the kilobytes of those that there are, copier w issues w, w + 4, ... (one too many is the last again;
        // behind it the LDS holds anything: columns of tokens that are never stored).  The wait leaves the copies of the last step in flight, so their number is a constant of the loop.
        const int pieces = (a.T - t0 < 16 * NTT ? a.T - t0 : 16 * NTT) * BAMD_B16_Q, ri = (pieces + 63) / 64, need = (ri + 3) / 4;
        auto copies = [&](auto nr_tag) {
            constexpr int NR = decltype(nr_tag)::value;
            uint32_t ro[NR], rd[NR];
#pragma unroll
            for (int r = 0; r < NR; ++r) {
                const int k = r * 4 + bw < ri ? r * 4 + bw : ri - 1, idx = k * 64 + lane, pi = idx < pieces ? idx : pieces - 1, tok = pi / BAMD_B16_Q;
                ro[r] = (uint32_t) (t0 + tok) * BAMD_B16_MEM + (uint32_t) (pi - tok * BAMD_B16_Q) * 16u; rd[r] = lds0 + REC0 + (uint32_t) k * 1024u;
            }
            auto copy_records = [&](int ci, int slot) {
                const void * src = uniform_ptr(a.blob16 + (size_t) (ci < nb ? ci : nb - 1) * BAMD_B16_STEP(a.T));
#pragma unroll
                for (int r = 0; r < NR; ++r) lds_dma16_s(src, ro[r], rd[r] + (uint32_t) slot * RS);
            };
            // records of 0 and the operands of 0 and 1 have landed when all but the last NR + 2 NW copies have; so it stays: at the end of step ci the records of ci + 1 (issued in
            // ci - 1) and the operands of ci + 2 (issued in ci - 2) have landed
            auto landed = [&] { asm volatile("s_waitcnt vmcnt(%0)" :: "n"(NR + 2 * NW) : "memory"); barrier(); };
            copy_records(0, 0); copy_weights(0, 0); copy_weights(1, 1); copy_records(1, 1); copy_weights(2, 2); copy_weights(3, 3);
            landed();
            barrier();
            for (int ci = 0, rs = 0, ws = 0; ci < nb; ++ci, rs = after(rs, 1, XF_RING), ws = after(ws, 1, XF_WRING)) {
                copy_records(ci + 2, after(rs, 2, XF_RING)); copy_weights(ci + 4, after(ws, 4, XF_WRING));
                if (Q6) barrier();
                landed();
            }
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");      // (no copy outlives the block)
        };
#define XF_NEED(N_) if (need <= N_) { copies(std::integral_constant<int, N_>()); return; }
        if constexpr (NTT == 2) { XF_NEED(1) XF_NEED(2) XF_NEED(3) XF_NEED(4) copies(std::integral_constant<int, 5>()); }       // up to 32 tokens
        else if constexpr (NTT == 3) { XF_NEED(5) XF_NEED(6) XF_NEED(7) copies(std::integral_constant<int, 8>()); }              // 33 to 48
        else { XF_NEED(8) XF_NEED(9) copies(std::integral_constant<int, 10>()); }                                              // 49 to 64
#undef XF_NEED
        return;
    }
    barrier();
    if (builder) {
        if constexpr (Q6) build6(smem + W0, 0, fr0); else build45(smem + W0, fr0);
        barrier();
        for (int ci = 0, ws = 0; ci < nb; ++ci) {
            const unsigned char * w = smem + W0 + ws * WS;
            ws = after(ws, 1, XF_WRING);
            const unsigned char * wn = smem + W0 + ws * WS;
            if constexpr (Q6) { build6(w, 1, fr1); barrier(); build6(wn, 0, fr0); }
            else build45(wn, (ci & 1) ? fr0 : fr1);
            barrier();
        }
        return;
    }
    barrier();
    for (int ci = 0, rs = 0, ws = 0; ci < nb; ++ci, rs = after(rs, 1, XF_RING), ws = after(ws, 1, XF_WRING)) {
        const unsigned char * recs = smem + REC0 + rs * RS, * w = smem + W0 + ws * WS;
        if (!active) { if (Q6) barrier(); }
        else if constexpr (Q6) {
            consume6(recs, w, fr0, std::integral_constant<int, 0>());
            barrier();
            consume6(recs, w, fr1, std::integral_constant<int, 1>());
        } else consume45(recs, w, (ci & 1) ? fr1 : fr0);
        barrier();
    }
    const int t = t0 + tt * 16 + m, row0 = rtg * 16 + 4 * g;
    if (!active || t >= a.T) return;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float v = ((acc[0][i] + acc[4][i]) + (acc[2][i] + acc[6][i])) + ((acc[1][i] + acc[5][i]) + (acc[3][i] + acc[7][i]));
        float val = v;
        if constexpr (!Q6) { const float mm = Q5 ? accm[0][i] : (accm[0][i] + accm[2][i]) + (accm[1][i] + accm[3][i]); val = v + mm; }
        if (row0 + i < a.nrows) {
            const size_t o = (size_t) t * a.ldo + row0 + i;
            a.out[o] = EPI == BAMD_EPI_ADD ? val + a.res[o] : EPI == BAMD_EPI_SILU_MUL ? v_silu(a.res[o]) * val : val;
        }
    }
}

template <int TYPE, int EPI, int NTT>
__global__ void __launch_bounds__(768) matmul_few_kernel(bamd_mma2_args a) { few_block<TYPE, EPI, NTT>(a, blockIdx.y); }
// Two products of the same tokens in one launch: the Q6_K one (`first` row tiles) in front, since its blocks take longer, then a Q4_K or Q5_K one.  By themselves queries and keys of the 8B shape
// are a round of 256 blocks and a quarter, values another quarter of one:
// a prompt of 37 tokens 5033 -> 4786 us (16 of 32 layers have such values)
template <int TYPE, int NTT>
__global__ void __launch_bounds__(768) matmul_few_two_kernel(bamd_mma2_args six, bamd_mma2_args a, int first) {
    if ((int) blockIdx.y < first) few_block<BAMD_Q6_K, BAMD_EPI_STORE, NTT>(six, blockIdx.y);
    else few_block<TYPE, BAMD_EPI_STORE, NTT>(a, blockIdx.y - first);
}

// ---- host side -----------------------------------------------------------------------------------------------------------------------------
static inline int x_row_blocks(int nrows_pad) { return (nrows_pad + 63) / 64; }
static unsigned long long * g_prefill_dbg = nullptr;      // -DX_TIMING builds: where the kernels of the next launches leave their phase clocks (bamd_prefill_dbg)
extern "C" __attribute__((visibility("default"))) void bamd_prefill_dbg(void * dev_buf) { g_prefill_dbg = (unsigned long long *) dev_buf; }
// bytes of the side table of a K-quant matrix [nrows_pad][K]: builder part first, the consumer part behind it (both 16-byte aligned)
size_t bamd_prefill_aux_bytes(int type, int nrows_pad, int K) {
    if ((type != BAMD_Q4_K && type != BAMD_Q5_K && type != BAMD_Q6_K) || (K & 255) || (nrows_pad & 7)) return 0;
    const size_t nb = (size_t) (K >> 8), rbk = (size_t) x_row_blocks(nrows_pad);
    // + two super-blocks of slack behind each table: the sixteen-wave kernel's last two staging calls read past the end of K
    return type == BAMD_Q6_K ? (rbk * nb + 2) * 8192 + (rbk * nb + 2) * 4 * X_CH6_RT : (rbk * nb + 2) * 4096 + (rbk * nb + 2) * X3_CHS;
}
static inline size_t x_ph_bytes(int type, int nrows_pad, int K) { return ((size_t) x_row_blocks(nrows_pad) * (size_t) (K >> 8) + 2) * (type == BAMD_Q6_K ? 8192 : 4096); }
void bamd_launch_prefill_aux(const void * w_stream, int type, int nrows_pad, int K, void * aux, hipStream_t s) {
    const int nb = K >> 8, nrt = x_row_blocks(nrows_pad) * 4;
    uint8_t * ph = (uint8_t *) aux, * ch = ph + x_ph_bytes(type, nrows_pad, K);
    const dim3 grid(nb, nrt);
    if (type == BAMD_Q6_K)      hipLaunchKernelGGL(prefill_aux_q6k_kernel, grid, dim3(64), 0, s, (const uint8_t *) w_stream, nrows_pad, nb, ph, ch);
    else if (type == BAMD_Q5_K) hipLaunchKernelGGL((prefill_aux_q4k_kernel<true>), grid, dim3(64), 0, s, (const uint8_t *) w_stream, nrows_pad, nb, ph, ch);
    else                        hipLaunchKernelGGL((prefill_aux_q4k_kernel<false>), grid, dim3(64), 0, s, (const uint8_t *) w_stream, nrows_pad, nb, ph, ch);
}
// the most dynamic LDS any launch below takes
static constexpr size_t x_max_lds() {
    size_t m = few_lds(BAMD_Q6_K, 4);
    for (const size_t v : { (size_t) X3_LDS_BYTES, few_lds(BAMD_Q4_K, 4), few_lds(BAMD_Q5_K, 4) }) m = v > m ? v : m;      // (bamd_prefill_wide.hip takes no more: asserted there)
    return m;
}
static bool x_takes(const void * kernel, size_t lds) { return hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int) lds) == hipSuccess; }
// 1 when the current device takes the matrix-core kernels' launches (159 328 B of dynamic LDS, up to 1024 threads): asked once per model load, before any side table is built, since a
// rejected launch would leave stale output behind a success code
int bamd_prefill_mfma_supported(void) {
    int dev = 0, lds = 0;
    if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&lds, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) != hipSuccess) { (void) hipGetLastError(); return 0; }
    if ((size_t) lds < x_max_lds()) return 0;
    if (!x_takes((const void *) matmul_mfma3_q4k_kernel<BAMD_EPI_STORE, false>, X3_LDS_BYTES) || !bamd_wide_supported() ||
        !x_takes((const void *) matmul_few_kernel<BAMD_Q6_K, BAMD_EPI_STORE, 4>, few_lds(BAMD_Q6_K, 4))) { (void) hipGetLastError(); return 0; }
    return 1;
}
// Token tiles (of 16) per block of the few-token kernel for this product, 0: one of the kernels with 64-row blocks.
// Up to 64 tokens and 16384 rows: whichever ends first.  The few-token kernel takes a start, and for every round of 256 blocks another and a time per super-block, which grows with the tokens whose records
// are copied; the other (64 rows a block: matmul_mfma3_q4k_kernel, for Q6_K matmul_wide_kernel's four waves) is in its first round up to 16384 rows, and behind that faster everywhere (of 1755 sizes).
// Constants in ns (token: tenths), fitted to 8190 sizes (three types, 6 to 64 tokens, 1024 to 16384 rows, K 1024 to 14336; weights from memory, launches one behind the other), of which this rule takes
// the slower kernel for 13 by more than 1.5 %, at most 4.6 %; of 1500 others, drawn at random, for 4, at most 3.0 %.  Prompts of eight 8B layers, 50 tokens 1327 -> 1247 us, 61 1365 -> 1296; six 7B ones in
// Q6_K, 26 942 -> 919, 48 1046 -> 1016.  Where the two part, us, few-token kernel and the other: Q4_K, K = 4096, 8192 rows 48 tokens 23.3 | 25.6, 64 26.4 | 26.1, 12288 rows 16 tokens
// 25.8 | 25.6, 32 tokens 28.5 | 25.6; 6144 rows x 3840 40 tokens 20.3 | 23.6; Q6_K, K = 4096, 4096 rows 40 tokens 16.5 | 27.2, 6144 rows 16 tokens 26.2 | 23.5, 40 30.7 | 27.5
struct x_cost { int extra, start[3], step[3], token[3], start64[3], step64[3]; };
static int x_few_tiles(int type, int nrows_pad, int nb, int T) {
    static const x_cost costs[3] = { { 1270, { 1950, 2230, 2490 }, { 335, 330, 334 }, { 30, 40, 43 }, { 3680, 3860, 3950 }, { 1346, 1335, 1355 } },         // Q4_K
                                     { 1140, { 2060, 2320, 2570 }, { 335, 283, 302 }, { 36, 58, 53 }, { 3530, 3630, 3430 }, { 1318, 1344, 1429 } },         // Q5_K
                                     { 1300, { 2250, 2670, 3080 }, { 541, 609, 751 }, { 54, 37, 10 }, { 3630, 4400, 4680 }, { 1243, 1429, 1637 } } };       // Q6_K
    if (T > 64 || nrows_pad > 16384) return 0;
    const x_cost & c = costs[type == BAMD_Q6_K ? 2 : type == BAMD_Q5_K ? 1 : 0];
    const int i = T <= 32 ? 0 : T <= 48 ? 1 : 2;
    const long few = c.extra + (long) ((nrows_pad + 15) / 16 + 255) / 256 * (c.start[i] + (10L * c.step[i] + (long) c.token[i] * T) * nb / 10);
    return few < c.start64[i] + (long) c.step64[i] * nb ? i + 2 : 0;
}
int bamd_prefill_few_tiles(int type, int nrows_pad, int K, int T) { return x_few_tiles(type, nrows_pad, K >> 8, T); }
size_t bamd_prefill_route(int type, int nrows_pad, int K, int T, int * few_tiles, size_t * most) {
    *few_tiles = x_few_tiles(type, nrows_pad, K >> 8, T); *most = x_max_lds();
    if (*few_tiles) return few_lds(type, *few_tiles);
    const int waves = bamd_prefill_tokfrag(type, nrows_pad, K, T);
    return waves ? bamd_wide_lds(type, T, waves) : X3_LDS_BYTES;
}
static bamd_mma2_args x_args(const bamd_few_side & w, int K, const void * blob16, int T, float * out, const float * res, int ldo) {
    const uint8_t * aux = (const uint8_t *) w.aux;
    return { (const uint8_t *) w.stream, aux, aux + x_ph_bytes(w.type, w.nrows_pad, K), out, res, (const uint8_t *) blob16, K, T, w.nrows, w.nrows_pad, ldo, g_prefill_dbg };
}
int bamd_launch_matmul_few_two(const bamd_few_side & six, float * out6, const bamd_few_side & w, float * out, int K, const void * blob16, int T, int ldo, hipStream_t s) {
    if (six.type != BAMD_Q6_K || (w.type != BAMD_Q4_K && w.type != BAMD_Q5_K) || ((six.nrows_pad | w.nrows_pad) & 7) || (K & 255) || !six.aux || !w.aux) return 1;
    const int ntt = x_few_tiles(w.type, w.nrows_pad, K >> 8, T);
    if (!ntt || x_few_tiles(six.type, six.nrows_pad, K >> 8, T) != ntt) return 1;
    const bamd_mma2_args a6 = x_args(six, K, blob16, T, out6, nullptr, ldo), a = x_args(w, K, blob16, T, out, nullptr, ldo);
    const int first = (six.nrows_pad + 15) / 16;
    const dim3 grid((T + 16 * ntt - 1) / (16 * ntt), first + (w.nrows_pad + 15) / 16);
#define XF2_LAUNCH(TYPE_, NTT_) hipLaunchKernelGGL((matmul_few_two_kernel<TYPE_, NTT_>), grid, dim3(768), std::max(few_lds(BAMD_Q6_K, NTT_), few_lds(TYPE_, NTT_)), s, a6, a, first)
#define XF2_TYPE(TYPE_) do { if (ntt == 2) XF2_LAUNCH(TYPE_, 2); else if (ntt == 3) XF2_LAUNCH(TYPE_, 3); else XF2_LAUNCH(TYPE_, 4); } while (0)
    if (w.type == BAMD_Q5_K) XF2_TYPE(BAMD_Q5_K); else XF2_TYPE(BAMD_Q4_K);
#undef XF2_TYPE
#undef XF2_LAUNCH
    return 0;
}
int bamd_launch_matmul_mfma2(const void * w_stream, const void * aux, int type, int nrows, int nrows_pad, int K, const void * blob16, int T, float * out, const float * res,
                             int epi, int ldo, hipStream_t s) {
    if ((type != BAMD_Q4_K && type != BAMD_Q5_K && type != BAMD_Q6_K) || (nrows_pad & 7) || (K & 255) || !aux) return 1;
    if (epi != BAMD_EPI_STORE && epi != BAMD_EPI_ADD && epi != BAMD_EPI_SILU_MUL) return 1;
    if ((epi != BAMD_EPI_STORE) != (res != nullptr)) return 1;
    const bamd_mma2_args a = x_args({ w_stream, aux, type, nrows, nrows_pad }, K, blob16, T, out, res, ldo);
    const dim3 grid((T + 63) / 64, x_row_blocks(nrows_pad));
    const dim3 grid3(grid.x, BAMD_PREFILL_CEILING == 2 ? (grid.y + 1) / 2 : grid.y);     // (ceiling build 2: every workgroup issues the MFMAs of two; timing only)
#define X3_LAUNCH(KERNEL, ...) do { \
        if (epi == BAMD_EPI_ADD)           hipLaunchKernelGGL((KERNEL<BAMD_EPI_ADD __VA_ARGS__>),      grid3, dim3(1024), X3_LDS_BYTES, s, a); \
        else if (epi == BAMD_EPI_SILU_MUL) hipLaunchKernelGGL((KERNEL<BAMD_EPI_SILU_MUL __VA_ARGS__>), grid3, dim3(1024), X3_LDS_BYTES, s, a); \
        else                               hipLaunchKernelGGL((KERNEL<BAMD_EPI_STORE __VA_ARGS__>),    grid3, dim3(1024), X3_LDS_BYTES, s, a); } while (0)
    if (const int ntt = x_few_tiles(type, nrows_pad, K >> 8, T)) {
#define XF_LAUNCH(TYPE_, NTT_) do { const dim3 gf((T + 16 * NTT_ - 1) / (16 * NTT_), (nrows_pad + 15) / 16); \
        if (epi == BAMD_EPI_ADD)           hipLaunchKernelGGL((matmul_few_kernel<TYPE_, BAMD_EPI_ADD, NTT_>),      gf, dim3(768), few_lds(TYPE_, NTT_), s, a); \
        else if (epi == BAMD_EPI_SILU_MUL) hipLaunchKernelGGL((matmul_few_kernel<TYPE_, BAMD_EPI_SILU_MUL, NTT_>), gf, dim3(768), few_lds(TYPE_, NTT_), s, a); \
        else                               hipLaunchKernelGGL((matmul_few_kernel<TYPE_, BAMD_EPI_STORE, NTT_>),    gf, dim3(768), few_lds(TYPE_, NTT_), s, a); } while (0)
#define XF_TYPE(TYPE_) do { if (ntt == 2) XF_LAUNCH(TYPE_, 2); else if (ntt == 3) XF_LAUNCH(TYPE_, 3); else XF_LAUNCH(TYPE_, 4); } while (0)
        if (type == BAMD_Q6_K)      XF_TYPE(BAMD_Q6_K);
        else if (type == BAMD_Q5_K) XF_TYPE(BAMD_Q5_K);
        else                        XF_TYPE(BAMD_Q4_K);
#undef XF_TYPE
#undef XF_LAUNCH
        return 0;
    }
    if (type == BAMD_Q6_K)      return 1;                         // (bamd_prefill_wide.hip)
    else if (type == BAMD_Q5_K) X3_LAUNCH(matmul_mfma3_q4k_kernel, , true);
    else                        X3_LAUNCH(matmul_mfma3_q4k_kernel, , false);
#undef X3_LAUNCH
    return 0;
}
