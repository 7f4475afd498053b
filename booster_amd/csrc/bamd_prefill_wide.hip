// bamd_prefill_wide.hip — the exact matrix-core mat-mul of many tokens (Q4_K / Q5_K / Q6_K x Q8_K): a wave owns 16 weight rows and up to 64 tokens.
//
// Reference: ggml_compute_forward_mul_mat with ne11 = T (ggml.c:12277-12492) over ggml_vec_dot_q{4,5,6}_K_q8_K (ggml-quants.c:6832 / :7400 / :8037).  Per (row, token) that is
// eight f32 chains (one per SIMD lane e) acc_e = fma(d_x d_y, isum_e, acc_e) over the super-blocks, four (Q5_K: one) chains of the min terms, and a sum tree at the end; the
// integer sums isum_e are exact on the matrix cores (one v_mfma_f32_16x16x32_f16 per e and 16 x 16 tile: f16 scale x quant times the int8 activations).
//
// What bounds it is the vector issue of a SIMD (measured, cycles: a vector instruction 4, this matrix instruction 16 of the matrix pipe and 8 of the same issue): 32 chain FMAs and 4
// products d_x d_y per tile and super-block, 16 + 4 for the min terms, twelve matrix instructions, and the expansion of the quants.  So
//   * a wave keeps all eight chains of 16 rows x 64 tokens (128 accumulators) and expands the quants of ITS rows once per super-block for four token tiles, in registers: no
//     fragment of weights goes through LDS, nothing is expanded twice, and no wave waits for another's expansion (the sixteen-wave kernel of bamd_prefill2.hip moves 413 KB
//     through LDS per 64 rows x 64 tokens and super-block, this one 145);
//   * rows are the N side: the lane that holds an accumulator holds its row's header too, so d comes out of the header that the scales come from;
//   * the min terms are a second pass over K with 64 accumulators of their own (they need 24 bytes per row and 36 per token and super-block): together they would spill;
//   * the only thing waves share is the token fragments, which lie in memory as the lanes read them (quantize_batch_kernel) and are copied to LDS a super-block ahead, one barrier
//     per super-block.  Quants and headers come through LDS too (private to the wave, two super-blocks ahead), which makes every request of the loop a counted copy; except with Q6_K on
//     eight waves, where two registers are kept in scratch memory and the compiler's wait for the one it reads back at the top of a super-block waits for the copies in flight as well.
// 2048 tokens, K = 4096, Q4_K, in a running prompt: 14336 rows 708 -> 523 us (343 -> 460 TFLOP/s), 6144 rows 312 -> 222, 4096 rows 216 -> 152; Q6_K, K = 14336, 4096 rows 880 -> 510.
// Per super-block of 128 rows x 64 tokens 2.1 us: by itself the 14336-row launch takes 471 us, 366 without the min pass, in Q5_K 459 and 394, in Q6_K 530.  Tried, when that was 2.3: the eight e on two waves (four waves per SIMD, half the registers): 3.0
// us; matrix instructions and chains pinned in turn: no faster; a loop without a seam between super-blocks: 2.5 us, 3.4 for Q6_K.
#include "bamd_device.h"
#include "bamd_mfma_common.h"
#include "bamd_kernels.h"
#include <type_traits>
#include <algorithm>

typedef _Float16 bamd_h2 __attribute__((ext_vector_type(2)));
union bamd_h2u { uint32_t u; bamd_h2 h; };

struct bamd_wide_args {
    const uint8_t * w;               // wave-stream records of the matrix (bamd_formats.h)
    const uint8_t * frag;            // token fragments (quantize_batch_kernel)
    float * out; const float * res;  // [T][ldo]
    const uint8_t * w2; float * out2;       // of the blocks z = 1
    int K, T, nrows, nrows_pad, ldo, epi;
};

// N kilobytes (2 or 4) that follow one another in memory and in LDS, 16 bytes per lane and kilobyte.  m0 is the compiler's to save (clobbered)
template <int N> __device__ __forceinline__ void wide_dma(const void * sbase, uint32_t voff, uint32_t lds_dst) {
    if (N == 4) asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1\n\tglobal_load_lds_dwordx4 %0, %1 offset:1024\n\tglobal_load_lds_dwordx4 %0, %1 offset:2048\n\tglobal_load_lds_dwordx4 %0, %1 offset:3072"
                             :: "v"(voff), "s"(sbase), "s"(lds_dst) : "memory", "m0");
    else if (N == 2) asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1\n\tglobal_load_lds_dwordx4 %0, %1 offset:1024" :: "v"(voff), "s"(sbase), "s"(lds_dst) : "memory", "m0");
    else asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" :: "v"(voff), "s"(sbase), "s"(lds_dst) : "memory", "m0");
}
__device__ __forceinline__ void wide_dma4(const void * sbase, uint32_t voff, uint32_t lds_dst) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dword %0, %1" :: "v"(voff), "s"(sbase), "s"(lds_dst) : "memory", "m0");
}
template <int TYPE> struct WideW {                        // a wave's 16 rows of one super-block in LDS, and the copies that bring them
    static constexpr int RECB = TYPE == BAMD_Q6_K ? 1680 : TYPE == BAMD_Q5_K ? BAMD_RECB_Q5K : BAMD_RECB_Q4K;
    static constexpr int HDR = TYPE == BAMD_Q6_K ? 3072 : TYPE == BAMD_Q5_K ? 2560 : 2048;       // 16 bytes per row: header (Q6_K: scales)
    static constexpr int SLOT = HDR + (TYPE == BAMD_Q6_K ? 512 : 256), COPIES = TYPE == BAMD_Q4_K ? 3 : 5;
};
constexpr int wide_tslot(int ntt) { return ntt * 8192 + 256; }
#define XW_MTOK 2304                                      /* min pass: token operands of a super-block: 64 tokens x 32 B, then 64 d_y */
constexpr int wide_mslot(int wv) { return 8 * XW_MTOK + wv * 2048 + 256; }      /* of eight super-blocks, and the headers of the block's rows */
template <int TYPE> constexpr size_t wide_main(int ntt, int wv) { return (size_t) 2 * wide_tslot(ntt) + (size_t) 3 * wv * WideW<TYPE>::SLOT; }
template <int TYPE> constexpr bool wide_mins_first(int ntt, int wv) {         // the min pass's first operands lie beside the product's
    return TYPE != BAMD_Q6_K && wide_main<TYPE>(ntt, wv) + wide_mslot(wv) <= 159328 && wide_main<TYPE>(ntt, wv) >= (size_t) wide_mslot(wv);
}
template <int TYPE> constexpr size_t wide_lds(int ntt, int wv) {
    const size_t m = wide_main<TYPE>(ntt, wv), s = wide_mslot(wv);
    return wide_mins_first<TYPE>(ntt, wv) ? m + s : TYPE == BAMD_Q6_K || m > 2 * s ? m : 2 * s;
}
static_assert(wide_lds<BAMD_Q4_K>(4, 8) <= 159328 && wide_lds<BAMD_Q5_K>(4, 8) <= 159328 && wide_lds<BAMD_Q6_K>(4, 8) <= 159328, "no more LDS than the load-time probe asks for");
template <int TYPE, int NTT, int WV>
__global__ void __launch_bounds__(64 * WV) matmul_wide_kernel(bamd_wide_args a) {
    constexpr bool Q4 = TYPE == BAMD_Q4_K, Q5 = TYPE == BAMD_Q5_K, Q6 = TYPE == BAMD_Q6_K;
    constexpr int RECB = WideW<TYPE>::RECB, WS = WideW<TYPE>::SLOT, HDR = WideW<TYPE>::HDR, TS = wide_tslot(NTT), NW = WideW<TYPE>::COPIES;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    if (blockIdx.z) { a.w = a.w2; a.out = a.out2; }
    const int lane = threadIdx.x & 63, wave = wave_id(), m = lane & 15, g = lane >> 4;
    const int nb = a.K >> 8, ntile = (a.T + 15) >> 4, tile0 = blockIdx.x * NTT;
    const int nrt = (a.nrows_pad + 15) >> 4, rt0 = blockIdx.y * WV + wave, rt = rt0 < nrt ? rt0 : nrt - 1;
    const uint32_t lds0 = (uint32_t) (size_t) (bamd_lds_vp) smem;
    const uint8_t * const dyp = a.frag + (size_t) ntile * nb * 8192, * const mnp = dyp + (size_t) ntile * nb * 64;
    auto tile_of = [&](int t) { return tile0 + t < ntile ? tile0 + t : ntile - 1; };

    // ---- copies.  Tokens: wave w brings kilobytes NTT w .. NTT w + NTT - 1 of the block's 8 NTT; d_y of the 64 tokens by every wave (the same bytes to the same place).
    // Tiles past the last one are the last one again (never stored).
    constexpr int NP = NTT * 8 / WV; constexpr bool RUN = 8 % NP == 0;      // kilobytes per wave; of one tile, and so one run
    const uint8_t * tsrc[RUN ? 1 : NP];
#pragma unroll
    for (int j = 0; j < (RUN ? 1 : NP); ++j) { const int k = wave * NP + j; tsrc[j] = uniform_ptr(a.frag + (size_t) tile_of(k >> 3) * nb * 8192 + (size_t) (k & 7) * 1024); }
    const uint32_t dyo = (uint32_t) tile_of(g < NTT ? g : NTT - 1) * (uint32_t) (nb * 64) + (uint32_t) m * 4u, l16 = (uint32_t) lane * 16u;
    const uint32_t tdst = lds0 + (uint32_t) (wave * NP) * 1024u;
    auto copy_tokens = [&](int ci, int slot) {
        const int c = ci < nb ? ci : nb - 1;
        const uint32_t d = tdst + (uint32_t) (slot * TS);
        if constexpr (!RUN) {
#pragma unroll
            for (int j = 0; j < NP; ++j) wide_dma<1>(tsrc[j] + (size_t) c * 8192, l16, d + (uint32_t) j * 1024u);
        } else if constexpr (NP == 8) { wide_dma<4>(tsrc[0] + (size_t) c * 8192, l16, d); wide_dma<4>(tsrc[0] + (size_t) c * 8192 + 4096, l16, d + 4096u); }
        else wide_dma<NP>(tsrc[0] + (size_t) c * 8192, l16, d);
        wide_dma4(dyp + (size_t) c * 64, dyo, lds0 + (uint32_t) (slot * TS + NTT * 8192));
    };
    // quants as 16-byte pieces [e][row] (in memory: [row group of 8][row][e]); a last tile of 8 (padded) rows takes its first record group twice (rows 8..15 are never stored)
    const uint8_t * const rec = uniform_ptr(a.w + (size_t) (2 * rt) * nb * RECB);
    const uint32_t group = (uint32_t) ((2 * rt + 1) * 8 < a.nrows_pad ? nb * RECB : 0);
    const uint32_t mrow = (uint32_t) (m >> 3) * group, q0 = mrow + (uint32_t) ((m & 7) * 8 + g) * 16u;
    const uint32_t hrow = (uint32_t) (lane >> 5) * group + (uint32_t) ((lane >> 2) & 7) * 16u + (uint32_t) (lane & 3) * 4u;      // row lane / 4, dword lane % 4 of its 16 bytes
    const uint32_t wdst = lds0 + (uint32_t) (2 * TS + wave * WS);
    auto copy_weights = [&](int ci, int slot) {
        const uint8_t * p = rec + (size_t) (ci < nb ? ci : nb - 1) * RECB;
        const uint32_t d = wdst + (uint32_t) (slot * WV * WS);
        wide_dma<1>(p, q0, d); wide_dma<1>(p, q0 + 64u, d + 1024u);
        if constexpr (Q4) wide_dma4(p + 1024, hrow, d + HDR);
        if constexpr (Q5) { wide_dma4(p + 1024, (uint32_t) lane * 4u, d + 2048u); wide_dma4(p + 1024, group + (uint32_t) lane * 4u, d + 2304u); wide_dma4(p + 1280, hrow, d + HDR); }
        if constexpr (Q6) {
            wide_dma<1>(p + 1024, mrow + (uint32_t) ((m & 7) * 4 + g) * 16u, d + 2048u);                          // high bits: pieces [e / 2][row]
            wide_dma4(p + 1536, hrow, d + HDR);
            wide_dma4(p + 1664, (uint32_t) ((lane >> 2) & 1) * group + (uint32_t) (lane & 3) * 4u, d + HDR + 256u);   // d of the 16 rows (eight dwords, again and again)
        }
    };
    // min pass: eight super-blocks at a time; a wave copies the token operands of one of them and the headers of its rows of all
    constexpr uint32_t HOFF = Q5 ? 1280u : 1024u;
    struct MinGeo { uint32_t tok[2], dy, hdr; };
    auto min_geo = [&](int ln) {
        MinGeo o;
#pragma unroll
        for (int j = 0; j < 2; ++j) { const int p = j * 64 + ln, t = p >> 5; o.tok[j] = (uint32_t) tile_of(t < NTT ? t : NTT - 1) * (uint32_t) (nb * 512) + (uint32_t) (p & 31) * 16u; }
        o.dy = (uint32_t) tile_of((ln >> 4) < NTT ? ln >> 4 : NTT - 1) * (uint32_t) (nb * 64) + (uint32_t) (ln & 15) * 4u;
        o.hdr = (uint32_t) (ln >> 5) * group + (uint32_t) ((ln >> 2) & 7) * 16u + (uint32_t) (ln & 3) * 4u;
        return o;
    };
    constexpr bool MF = wide_mins_first<TYPE>(NTT, WV);
    auto mslot = [](int slot) { return (uint32_t) (MF ? (slot ? 0 : wide_main<TYPE>(NTT, WV)) : slot * wide_mslot(WV)); };
    auto copy_mins = [&](int c8, int slot, const MinGeo & mg) {
        const uint32_t h = lds0 + mslot(slot) + (uint32_t) (8 * XW_MTOK + wave * 2048);
#pragma unroll
        for (int j = 0; j < 8 / WV; ++j) {
            const int k = wave * (8 / WV) + j, c = c8 * 8 + k < nb ? c8 * 8 + k : nb - 1;
            const uint32_t d = lds0 + mslot(slot) + (uint32_t) (k * XW_MTOK);
            wide_dma<1>(mnp + (size_t) c * 512, mg.tok[0], d); wide_dma<1>(mnp + (size_t) c * 512, mg.tok[1], d + 1024u); wide_dma4(dyp + (size_t) c * 64, mg.dy, d + 2048u);
        }
#pragma unroll
        for (int k = 0; k < 8; ++k) wide_dma4(rec + (size_t) (c8 * 8 + k < nb ? c8 * 8 + k : nb - 1) * RECB + HOFF, mg.hdr, h + (uint32_t) k * 256u);
    };
    auto publish = [&](auto left) { asm volatile("s_waitcnt vmcnt(%0)" :: "n"(decltype(left)::value) : "memory"); __builtin_amdgcn_s_barrier(); asm volatile("" ::: "memory"); };
    bamd_f4 acc[NTT][8];
#pragma unroll
    for (int t = 0; t < NTT; ++t)
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[t][e] = (bamd_f4) { 0.f, 0.f, 0.f, 0.f };
    const bamd_f4 z = { 0.f, 0.f, 0.f, 0.f };
    const bamd_h2 k1024 = { (_Float16) -1024.f, (_Float16) -1024.f }, k1056 = { (_Float16) -1056.f, (_Float16) -1056.f }, k1152 = { (_Float16) -1152.f, (_Float16) -1152.f };
    auto pair_of = [](uint32_t bytes, uint32_t sel) { bamd_h2u c; c.u = __builtin_amdgcn_perm(0x64646464u, bytes, sel); return c.h; };       // two bytes as 1024 + byte, f16
    // (constants in registers, unknown to the compiler: one v_and_or_b32, which takes no literals, for v_and_b32 and v_or_b32 with literals; 32 of 265 vector instructions a super-block,
    // the product's loop 3290 -> 3134 cycles, 14336 rows x 2048 tokens x 4096 499 -> 484 us)
    uint32_t k6400 = 0x64006400u, low = 0x000f000fu, high = 0x00f000f0u;
    if constexpr (Q4) { asm volatile("" : "+v"(k6400)); asm volatile("" : "+s"(low), "+s"(high)); }
    auto plus1024 = [&](uint32_t v, uint32_t mask) { bamd_h2u c; c.u = (v & mask) | k6400; return c.h; };
    union Frag { bamd_h2 h[4]; bamd_h8 v; };
    const uint32_t upper = 0u - (uint32_t) (g >> 1);              // (a mask, no branch)
    bamd_h2 s0, n0, s1, n1, sl0, sl1; uint32_t sc6[2];
    auto scales_of = [&](const unsigned char * w) -> float {
        if constexpr (Q6) {
#pragma unroll
            for (int h = 0; h < 2; ++h) sc6[h] = *(const uint32_t *) (w + HDR + m * 16 + (h * 2 + (g >> 1)) * 4) >> (16 * (g & 1));      // of sub-blocks 2g, 2g+1 in e-half h
            return h2f(*(const unsigned short *) (w + HDR + 256 + m * 2));
        } else {
            const uint4 hd = *(const uint4 *) (w + HDR + m * 16);
            // scales of sub-blocks 2g, 2g+1 (ggml-quants.c:6928-6933), as {s, -1024 s}; Q4_K's high nibbles stay in place (16 n): s / 16
            const uint32_t b = ((upper & ((hd.w & 0x0f0f0f0fu) | ((hd.y >> 2) & 0x30303030u))) | (~upper & hd.y & 0x3f3f3f3fu)) >> (16 * (g & 1));
            s0 = pair_of(b, 0x04000400u) + k1024; s1 = pair_of(b, 0x04010401u) + k1024;
            n0 = s0 * k1024;
            if constexpr (Q5) n1 = s1 * k1024;
            else { n1 = s1 * (bamd_h2) { (_Float16) -64.f, (_Float16) -64.f }; s1 = s1 * (bamd_h2) { (_Float16) 0.0625f, (_Float16) 0.0625f }; }
            return h2f(hd.x & 0xffffu);
        }
    };
    auto half_scales = [&](int h) {                               // Q6_K: split sc = sa + sl with sa = sc & ~15, sl = sc & 15
        const uint32_t hi = (sc6[h] ^ 0x80808080u) & 0xf0f0f0f0u, lo = sc6[h] & 0x0f0f0f0fu;
        s0 = pair_of(hi, 0x04000400u) + k1152; s1 = pair_of(hi, 0x04010401u) + k1152;
        sl0 = pair_of(lo, 0x04000400u) + k1024; sl1 = pair_of(lo, 0x04010401u) + k1024;
    };
    struct Raw { uint32_t q, q2, h; };
    auto raw_of = [&](const unsigned char * w, int e) {
        Raw r = { 0u, 0u, 0u };
        if constexpr (Q6) {
            const uint2 q = *(const uint2 *) (w + e * 256 + m * 16 + (g >> 1) * 8); r.q = q.x; r.q2 = q.y;
            r.h = *(const uint32_t *) (w + 2048 + (e >> 1) * 256 + m * 16 + (e & 1) * 8 + (g >> 1) * 4);
        } else {
            r.q = *(const uint32_t *) (w + e * 256 + m * 16 + g * 4);
            if constexpr (Q5) r.h = *(const uint32_t *) (w + 2048 + (m >> 3) * 256 + (m & 7) * 32 + e * 4);
        }
        return r;
    };
    auto build = [&](const Raw & r, int e, Frag & f, Frag & fl) {  // halves in the order 0, 2, 1, 3 of their dword, as the tokens' are
        if constexpr (Q6) {                                       // scale x (q - 32) reaches 4096: two fragments, (q - 32) sa and (q - 32) sl, both exact
            if ((e & 3) == 0) half_scales(e >> 2);
            const uint32_t sh = 4u * (uint32_t) (g & 1);
            const uint32_t uA = (__builtin_amdgcn_alignbit(r.h, r.h, (28u + sh) & 31u) & 0x30303030u) | ((r.q >> sh) & 0x0f0f0f0fu);
            const uint32_t uB = (__builtin_amdgcn_alignbit(r.h, r.h, (30u + sh) & 31u) & 0x30303030u) | ((r.q2 >> sh) & 0x0f0f0f0fu);
            const bamd_h2 v0 = pair_of(uA, 0x04020400u) + k1056, v1 = pair_of(uA, 0x04030401u) + k1056, v2 = pair_of(uB, 0x04020400u) + k1056, v3 = pair_of(uB, 0x04030401u) + k1056;
            f.h[0] = v0 * s0; f.h[1] = v1 * s0; f.h[2] = v2 * s1; f.h[3] = v3 * s1;
            fl.h[0] = v0 * sl0; fl.h[1] = v1 * sl0; fl.h[2] = v2 * sl1; fl.h[3] = v3 * sl1;
        } else {                                                  // (1024 + n) s - 1024 s = n s, one rounding, exact
            if constexpr (Q5) {
                const uint32_t q = r.h >> (2 * g);
                const uint32_t lo = (r.q & 0x0f0f0f0fu) | ((q & 0x01010101u) << 4), hi = ((r.q >> 4) & 0x0f0f0f0fu) | (((q >> 1) & 0x01010101u) << 4);
                f.h[0] = __builtin_elementwise_fma(pair_of(lo, 0x04020400u), s0, n0); f.h[1] = __builtin_elementwise_fma(pair_of(lo, 0x04030401u), s0, n0);
                f.h[2] = __builtin_elementwise_fma(pair_of(hi, 0x04020400u), s1, n1); f.h[3] = __builtin_elementwise_fma(pair_of(hi, 0x04030401u), s1, n1);
            } else {
                const uint32_t w8 = r.q >> 8;
                f.h[0] = __builtin_elementwise_fma(plus1024(r.q, low), s0, n0); f.h[1] = __builtin_elementwise_fma(plus1024(w8, low), s0, n0);
                f.h[2] = __builtin_elementwise_fma(plus1024(r.q, high), s1, n1); f.h[3] = __builtin_elementwise_fma(plus1024(w8, high), s1, n1);
            }
        }
    };
    bamd_h8 B[2][NTT]; Frag A[2], Al[2]; bamd_f4 S[2][NTT]; float D[NTT][4]; Raw raw[2];
    if constexpr (MF) copy_mins(0, 0, min_geo(lane));
    copy_weights(0, 0); copy_tokens(0, 0); copy_weights(1, 1);
    publish(std::integral_constant<int, NW>());
    const unsigned char * w = smem + 2 * TS + wave * WS;
    float dx = scales_of(w);
    raw[0] = raw_of(w, 0); raw[1] = raw_of(w, 1);
    build(raw[0], 0, A[0], Al[0]);
#pragma unroll
    for (int t = 0; t < NTT; ++t) {
        S[1][t] = z;
#pragma unroll
        for (int i = 0; i < 4; ++i) D[t][i] = 0.f;
    }
    int wnext = 1, wcopy = 2, ci = 0;                             // weight slots of ci + 1 and of ci + 2
    do {
        const unsigned char * tok = smem + (ci & 1) * TS + lane * 16, * wn = smem + 2 * TS + (wnext * WV + wave) * WS;
        publish(std::integral_constant<int, NW>());               // the tokens of ci are here (in flight: the weights of ci + 1); everyone is done with those of ci - 1
#pragma unroll
        for (int t = 0; t < NTT; ++t) B[0][t] = *(const bamd_h8 *) (tok + t * 8192);
#pragma unroll
        for (int t = 0; t < NTT; ++t)
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[t][7][i] = fmaf(D[t][i], S[1][t][i], acc[t][7][i]);      // of ci - 1
#pragma unroll
        for (int t = 0; t < NTT; ++t) {
            const bamd_f4 dy = *(const bamd_f4 *) (tok - lane * 16 + g * 16 + NTT * 8192 + t * 64);
#pragma unroll
            for (int i = 0; i < 4; ++i) D[t][i] = dy[i] * dx;
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            if (e < 7) {
#pragma unroll
                for (int t = 0; t < NTT; ++t) B[(e + 1) & 1][t] = *(const bamd_h8 *) (tok + t * 8192 + (e + 1) * 1024);
            } else {                                              // the weights of ci + 1 have landed
                asm volatile("s_waitcnt vmcnt(%0)" :: "n"(NP + 1 + NW) : "memory");
                dx = scales_of(wn); raw[0] = raw_of(wn, 0); raw[1] = raw_of(wn, 1);
            }
            if (e > 0 && e < 7) raw[(e + 1) & 1] = raw_of(w, e + 1);
#pragma unroll
            for (int t = 0; t < NTT; ++t) S[e & 1][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(B[e & 1][t], A[e & 1].v, z, 0, 0, 0);
            if constexpr (Q6) {
#pragma unroll
                for (int t = 0; t < NTT; ++t) S[e & 1][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(B[e & 1][t], Al[e & 1].v, S[e & 1][t], 0, 0, 0);
            }
            if (e == 1) copy_tokens(ci + 1, (ci + 1) & 1);
            if (e == 3) copy_weights(ci + 2, wcopy);
            build(raw[(e + 1) & 1], (e + 1) & 7, A[(e + 1) & 1], Al[(e + 1) & 1]);
            if (e > 0) {
#pragma unroll
                for (int t = 0; t < NTT; ++t)
#pragma unroll
                    for (int i = 0; i < 4; ++i) acc[t][e - 1][i] = fmaf(D[t][i], S[(e - 1) & 1][t][i], acc[t][e - 1][i]);
            }
            __builtin_amdgcn_sched_group_barrier(0x100, NTT + 2, 0);
#pragma unroll
            for (int t = 0; t < NTT * (Q6 ? 2 : 1); ++t) { __builtin_amdgcn_sched_group_barrier(0x2, Q6 ? 3 : 4, 0); __builtin_amdgcn_sched_group_barrier(0x8, 1, 0); }
            __builtin_amdgcn_sched_barrier(0);
        }
        w = wn; wnext = wcopy; wcopy = wcopy == 2 ? 0 : wcopy + 1;
    } while (++ci < nb);
#pragma unroll
    for (int t = 0; t < NTT; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[t][7][i] = fmaf(D[t][i], S[1][t][i], acc[t][7][i]);
    // (the lane again, unknown to the compiler: what the rest derives from it would be kept in registers through the loop above)
    int ln = threadIdx.x & 63; asm volatile("" : "+v"(ln));
    const int m2 = ln & 15, g2 = ln >> 4;
    const int row = rt0 * 16 + m2;
    float val[NTT][4], res[NTT][4];                               // hsum_float_8 over e, in the reference's order
#pragma unroll
    for (int t = 0; t < NTT; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            val[t][i] = ((acc[t][0][i] + acc[t][4][i]) + (acc[t][2][i] + acc[t][6][i])) + ((acc[t][1][i] + acc[t][5][i]) + (acc[t][3][i] + acc[t][7][i]));
            asm volatile("" : "+v"(val[t][i]));                   // (summed here: left alone the compiler carries all eight through the min pass)
        }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    publish(std::integral_constant<int, 0>());                    // no copy is in flight, nobody reads the LDS any more
    if (a.epi != BAMD_EPI_STORE) {
#pragma unroll
        for (int t = 0; t < NTT; ++t)
#pragma unroll
            for (int i = 0; i < 4; ++i) { const int tk = (tile0 + t) * 16 + 4 * g2 + i; res[t][i] = a.res[(size_t) (tk < a.T ? tk : a.T - 1) * a.ldo + (row < a.nrows ? row : 0)]; }
    }
    if constexpr (!Q6) {
        // ---- min terms: prod_l = m_2l S_2l + m_2l+1 S_2l+1 of sub-block pair l, chained over the super-blocks as fma(-d_y dmin, prod_l, acc_l) for each l (Q5_K: one chain of the
        // sum over l, product and sum rounded apart).  |S| <= 4064 is no f16: S = (S & ~1) + (S & 1), both exact.  Lane group g of v_mfma_f32_16x16x16_f16 holds pair g of the
        // tokens; the rows' operand of chain l is zero in the other groups
        const MinGeo geo = min_geo(ln);
        const uint32_t up2 = 0u - (uint32_t) (g2 >> 1);
        const int n8 = (nb + 7) >> 3;
        constexpr int NL = Q5 ? 1 : 4;
        uint32_t ml[4];
#pragma unroll
        for (int l = 0; l < 4; ++l) ml[l] = g2 == l ? ~0u : 0u;
        bamd_f4 accm[NTT][NL];
#pragma unroll
        for (int t = 0; t < NTT; ++t)
#pragma unroll
            for (int l = 0; l < NL; ++l) accm[t][l] = z;
        if constexpr (!MF) copy_mins(0, 0, geo);
        int c8 = 0;
        do {
            publish(std::integral_constant<int, 0>());
            if (c8 + 1 < n8) copy_mins(c8 + 1, (c8 + 1) & 1, geo);
            const unsigned char * base = smem + mslot(c8 & 1);
            const int n = nb - c8 * 8 < 8 ? nb - c8 * 8 : 8;
            const unsigned char * tk = base + g2 * 128 + m2 * 8, * dk = base + 2048 + g2 * 16, * hk = base + 8 * XW_MTOK + wave * 2048 + m2 * 16;
            // the operands of super-block k + 1 are requested in front of the chains of k (behind the last one: the LDS that follows, unused)
            struct Mins { uint4 hd; bamd_h4 S[NTT]; bamd_f4 dy[NTT]; } o[2];
            auto request = [&](int k, Mins & r) {
                r.hd = *(const uint4 *) (hk + k * 256);
#pragma unroll
                for (int t = 0; t < NTT; ++t) { r.S[t] = *(const bamd_h4 *) (tk + k * XW_MTOK + t * 512); r.dy[t] = *(const bamd_f4 *) (dk + k * XW_MTOK + t * 64); }
            };
            auto chains = [&](const Mins & r) {
                const float dm = h2f(r.hd.x >> 16);
                const uint32_t mw = ((up2 & (((r.hd.w >> 4) & 0x0f0f0f0fu) | ((r.hd.z >> 2) & 0x30303030u))) | (~up2 & r.hd.z & 0x3f3f3f3fu)) >> (16 * (g2 & 1));
                bamd_h2u mm; mm.h = pair_of(mw, 0x04010400u) + k1024;
                union { uint32_t u[2]; bamd_h4 h; } M[NL];
#pragma unroll
                for (int l = 0; l < NL; ++l) M[l].u[0] = M[l].u[1] = Q5 ? mm.u : mm.u & ml[l];
                bamd_f4 pm[2][NL];
#pragma unroll
                for (int t = 0; t <= NTT; ++t) {                  // the chains of a token tile beside the matrix instructions of the next
                    if (t < NTT) {
#pragma unroll
                        for (int l = 0; l < NL; ++l) pm[t & 1][l] = __builtin_amdgcn_mfma_f32_16x16x16f16(r.S[t], M[l].h, z, 0, 0, 0);
                    }
                    if (t > 0) {
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            const float dd = (-r.dy[t - 1][i]) * dm;
                            if constexpr (Q5) { const float p = dd * pm[(t - 1) & 1][0][i]; accm[t - 1][0][i] = accm[t - 1][0][i] + p; }
                            else {
#pragma unroll
                                for (int l = 0; l < NL; ++l) accm[t - 1][l][i] = fmaf(dd, pm[(t - 1) & 1][l][i], accm[t - 1][l][i]);
                            }
                        }
                    }
                    if (t > 0 && t < NTT) {
#pragma unroll
                        for (int l = 0; l < NL; ++l) { __builtin_amdgcn_sched_group_barrier(0x8, 1, 0); __builtin_amdgcn_sched_group_barrier(0x2, 5, 0); }
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
            };
            request(0, o[0]);
            int k = 0;
            do {
                request(1, o[1]); __builtin_amdgcn_sched_barrier(0);
                chains(o[0]);
                if (++k == n) break;
                request(2, o[0]); __builtin_amdgcn_sched_barrier(0);
                chains(o[1]);
                tk += 2 * XW_MTOK; dk += 2 * XW_MTOK; hk += 512;
            } while (++k < n);
        } while (++c8 < n8);
#pragma unroll
        for (int t = 0; t < NTT; ++t)
#pragma unroll
            for (int i = 0; i < 4; ++i) val[t][i] = val[t][i] + (Q5 ? accm[t][0][i] : (accm[t][0][i] + accm[t][NL > 2 ? 2 : 0][i]) + (accm[t][NL > 2 ? 1 : 0][i] + accm[t][NL > 2 ? 3 : 0][i]));
    }
    if (row >= a.nrows) return;
#pragma unroll
    for (int t = 0; t < NTT; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int tk = (tile0 + t) * 16 + 4 * g2 + i;
            if (tk >= a.T) continue;
            const float v = val[t][i];
            a.out[(size_t) tk * a.ldo + row] = a.epi == BAMD_EPI_ADD ? v + res[t][i] : a.epi == BAMD_EPI_SILU_MUL ? v_silu(res[t][i]) * v : v;
        }
}

// ---- host side -----------------------------------------------------------------------------------------------------------------------------
size_t bamd_tokfrag_bytes(int T, int K) { return (size_t) ((T + 15) / 16) * (size_t) (K >> 8) * (8192 + 64 + 512); }
// token tiles (of 16) per block: as few blocks as 64 tokens each allow, and the tiles spread over them
static int wide_tiles(int T) { const int tiles = (T + 15) / 16, blocks = (tiles + 3) / 4; return std::max(2, (tiles + blocks - 1) / blocks); }
static int wide_rounds(int nrows_pad, int T, int waves) { return (((T + 15) / 16 + wide_tiles(T) - 1) / wide_tiles(T) * (((nrows_pad + 15) / 16 + waves - 1) / waves) + 255) / 256; }
int bamd_prefill_tokfrag(int type, int nrows_pad, int K, int T) {
    if (bamd_prefill_few_tiles(type, nrows_pad, K, T)) return 0;
    // Both sides by their rounds of 256 blocks, one block per CU, and a round's time at K = 4096 in us (it grows with K alike): 64 x 64 on sixteen waves 26; here 26 | 32 | 38 with two,
    // three, four token tiles.  Q5_K and other K go by the same line: of 143 sizes each of Q4_K and Q5_K (65 to 2048 tokens, 1024 to 14336 rows, K from 2048 to 14336) it takes the slower
    // kernel by more than a hundredth nowhere.  Measured, 4096-row model: 14336 rows 96 tokens 50 | 35, 128 tokens 52 | 41, 200 tokens 97 | 77; 6144 rows 128 tokens 27 | 36, 200 tokens 50 | 38; 4096
    // rows 256 tokens 29 | 37, 512 tokens 54 | 41.  Q6_K, four waves against eight: 1024 rows 512 tokens 31 | 39, K = 14336 4096 rows 256 tokens 101 | 121, 512 tokens 198 | 136
    if (type == BAMD_Q6_K) return wide_rounds(nrows_pad, T, 8) * 100 <= wide_rounds(nrows_pad, T, 4) * 77 ? 8 : 4;
    static const int round[3] = { 26, 32, 38 };
    return wide_rounds(nrows_pad, T, 8) * round[wide_tiles(T) - 2] < (((T + 63) / 64) * ((nrows_pad + 63) / 64) + 255) / 256 * 26 ? 8 : 0;
}
size_t bamd_wide_lds(int type, int T, int waves) {
    const int n = wide_tiles(T);
    return type == BAMD_Q6_K ? wide_lds<BAMD_Q6_K>(n, waves) : type == BAMD_Q5_K ? wide_lds<BAMD_Q5_K>(n, waves) : wide_lds<BAMD_Q4_K>(n, waves);
}
bool bamd_wide_supported(void) {
    auto takes = [](const void * k, size_t lds) { return hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int) lds) == hipSuccess; };
    return takes((const void *) matmul_wide_kernel<BAMD_Q4_K, 4, 8>, wide_lds<BAMD_Q4_K>(4, 8)) && takes((const void *) matmul_wide_kernel<BAMD_Q6_K, 4, 8>, wide_lds<BAMD_Q6_K>(4, 8));
}
int bamd_launch_matmul_wide(const void * w_stream, int type, int nrows, int nrows_pad, int K, const void * frag, int T, float * out, const float * res, int epi, int ldo, int waves, hipStream_t s, const void * w2, float * out2) {
    if ((type != BAMD_Q4_K && type != BAMD_Q5_K && type != BAMD_Q6_K) || (nrows_pad & 7) || (K & 255) || K <= 0 || T <= 0 || nrows <= 0) return 1;
    if (epi != BAMD_EPI_STORE && epi != BAMD_EPI_ADD && epi != BAMD_EPI_SILU_MUL) return 1;
    if ((epi != BAMD_EPI_STORE) != (res != nullptr) || (w2 != nullptr) != (out2 != nullptr) || (w2 && epi != BAMD_EPI_STORE) || (waves != 8 && (waves != 4 || type != BAMD_Q6_K))) return 1;
    const bamd_wide_args a = { (const uint8_t *) w_stream, (const uint8_t *) frag, out, res, (const uint8_t *) w2, out2, K, T, nrows, nrows_pad, ldo, epi };
    const int n = wide_tiles(T);
    const dim3 grid(((T + 15) / 16 + n - 1) / n, ((nrows_pad + 15) / 16 + waves - 1) / waves, w2 ? 2 : 1);
#define XW_W(TYPE_, N_, WV_) hipLaunchKernelGGL((matmul_wide_kernel<TYPE_, N_, WV_>), grid, dim3(64 * WV_), wide_lds<TYPE_>(N_, WV_), s, a)
#define XW_N(TYPE_, WV_) do { if (n == 2) XW_W(TYPE_, 2, WV_); else if (n == 3) XW_W(TYPE_, 3, WV_); else XW_W(TYPE_, 4, WV_); } while (0)
    if (type == BAMD_Q4_K) XW_N(BAMD_Q4_K, 8); else if (type == BAMD_Q5_K) XW_N(BAMD_Q5_K, 8); else if (waves == 8) XW_N(BAMD_Q6_K, 8); else XW_N(BAMD_Q6_K, 4);
#undef XW_N
#undef XW_W
    return 0;
}
