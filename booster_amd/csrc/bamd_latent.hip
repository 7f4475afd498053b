// bamd_latent.hip — latent attention: per position one vector c of kv_rank values is cached (64-position pages); keys and values are linear in it.
//   prompts: the latents of the sequence are unpacked once per step into keys and transposed values (two dense products) and a flash kernel runs per head — 64 keys per
//     pass, scores, running maximum and sums in 32-bit, the weights as two bfloat16 terms (value + remainder) in front of the matrix cores;
//   decoding: the query is carried into the latent space (q W_uk per head) and all heads of a sequence share the cached rows: one pass over the cache in `splits`
//     parts, partial sums combined, then the value up-projection per head.
// A sink enters as the first key's place in the running maximum and sum (weight exp(sink), no value); a gate multiplies each head by sigmoid of its own projection.
#include "bamd_dense_device.h"
#include <algorithm>
#include <math.h>

// ---- the cache --------------------------------------------------------------------------------------------------------------------------------------
template <typename T> __device__ __forceinline__ void latent_store_row(const bamd_batch_dev & b, const bamd_latent_args & a, int row, float * red) {
    const bamd_entry e = b.ent[b.row_entry[row]];
    const int p = e.pos0 + (row - e.row0);
    const float * c = a.in + (size_t) row * a.ld + a.c_off;
    float v[1] = { 0.f };
    for (int i = threadIdx.x; i < a.R; i += blockDim.x) v[0] += c[i] * c[i];
    block_sum<1>(v, red);
    const float r = 1.0f / sqrtf(v[0] / (float) a.R + a.eps);
    T * d = (T *) a.cache + ((size_t) b.pages[(size_t) e.seq * b.max_pages + p / BAMD_PAGE] * BAMD_PAGE + p % BAMD_PAGE) * a.Rp;
    for (int i = threadIdx.x; i < a.Rp; i += blockDim.x) d[i] = to_act<T>(i < a.R ? c[i] * r * a.c_norm[i] : 0.f);
}
template <typename T> __global__ void __launch_bounds__(256) latent_store_kernel(bamd_batch_dev b, bamd_latent_args a) {
    __shared__ float red[16];
    latent_store_row<T>(b, a, blockIdx.x, red);
}
// one block per 64 rows of the destination = one page of a sequence
template <typename T> __global__ void __launch_bounds__(256) latent_gather_kernel(bamd_batch_dev b, bamd_latent_args a, const int32_t * k_entry, T * dst) {
    const bamd_entry e = b.ent[k_entry[blockIdx.x]];
    const int pg = blockIdx.x - e.kbase / BAMD_PAGE, len = e.pos0 + e.n, n = min(BAMD_PAGE, len - pg * BAMD_PAGE);
    const bamd_u4 * src = (const bamd_u4 *) ((const T *) a.cache + (size_t) b.pages[(size_t) e.seq * b.max_pages + pg] * BAMD_PAGE * a.Rp);
    bamd_u4 * d = (bamd_u4 *) (dst + (size_t) blockIdx.x * BAMD_PAGE * a.Rp);
    const int per = a.Rp * (int) sizeof(T) / 16;
    for (int i = threadIdx.x; i < BAMD_PAGE * per; i += 256) d[i] = i < n * per ? src[i] : bamd_u4{ 0, 0, 0, 0 };
}

// ---- prompts ----------------------------------------------------------------------------------------------------------------------------------------
// ND: head size in 32s (queries, keys and values); RT: 16-row query tiles per wave; four waves.  A wave's pass is a chain — keys, scores, maxima, weights through LDS, values — which only other
// waves fill: two blocks fit a CU's LDS with bfloat16 heads of up to 128, and registers are held to the half that lets both be there.  Maxima of sixteen lanes by data-parallel moves, sums added
// up once at the end, sums rescaled only in passes that move a maximum.  2048 tokens x 32 heads x 128: 211 us; moves for permutes of LDS and fewer rescales 158; two blocks per CU 146; paired 141; (on another card) exponents as fused products 133 -> 129
template <typename T, int ND, int RT>
__global__ void __launch_bounds__(256, sizeof(T) == 2 && ND <= 4 ? 2 : 1) latent_prompt_kernel(bamd_batch_dev b, bamd_latent_args a, const bamd_qtile * tiles, int n_heads, const T * kmat, const T * vt, int ldv) {
    constexpr int D = ND * 32, NV = ND * 2, KS = D + 16 / sizeof(T), VS = 64 + 16 / sizeof(T), NP = sizeof(T) == 2 ? 2 : 1;     // NP: terms of a weight
    constexpr int PIECES = 64 * D * (int) sizeof(T) / 16;
    extern __shared__ __align__(16) unsigned char lds[];
    T * Ks = (T *) lds, * Vs = Ks + 64 * KS, * Ps = Vs + D * VS;                 // Ps: per wave [NP][16 RT][VS]
    const int h = blockIdx.x % n_heads;
    const bamd_qtile qt = tiles[paired_tile(n_heads)];
    const bamd_entry e = b.ent[qt.entry];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, lr = lane & 15, lq = lane >> 4;
    T * P = Ps + (size_t) wave * NP * 16 * RT * VS;
    const int r0 = qt.q0 + wave * 16 * RT;                         // first query of this wave, counted in the entry
    Frag<T> q[RT][ND];
#pragma unroll
    for (int i = 0; i < RT; ++i) {
        int r = r0 + i * 16 + lr; r = r < e.n ? r : e.n - 1;
        const float * src = a.in + (size_t) (e.row0 + r) * a.ld + a.q_off + h * D;
#pragma unroll
        for (int k = 0; k < ND; ++k) {
            const bamd_v4 x = *(const bamd_v4 *) (src + k * 32 + lq * 8), y = *(const bamd_v4 *) (src + k * 32 + lq * 8 + 4);
#pragma unroll
            for (int j = 0; j < 4; ++j) { q[i][k].set(j, x[j]); q[i][k].set(4 + j, y[j]); }
        }
    }
    bamd_v4 o[RT][NV]; float m[RT][4], l[RT][4];
    // Maxima and the sink are kept times log2(e).  An exponent is one fused product and difference with the maximum: the product of a score is not rounded, and what the maximum was rounded
    // by is common to the keys and the sink
    const float l2e = 1.4426950408889634f, scale = a.scale * l2e, snk = a.sink ? a.sink[h] * l2e : -INFINITY;
    const float one = !a.sink ? 0.f : fabsf(snk) < INFINITY ? __builtin_amdgcn_exp2f(fmaf(a.sink[h], l2e, -snk)) : 1.f;
#pragma unroll
    for (int i = 0; i < RT; ++i) {
#pragma unroll
        for (int k = 0; k < 4; ++k) { m[i][k] = snk; l[i][k] = lr == 0 ? one : 0.f; }
#pragma unroll
        for (int j = 0; j < NV; ++j) o[i][j] = bamd_v4{ 0, 0, 0, 0 };
    }
    const int q_hi = min(qt.q0 + 64 * RT, e.n) - 1, len = e.pos0 + q_hi + 1;    // keys 0 .. len - 1
    const int w_hi = e.pos0 + min(r0 + 16 * RT, e.n) - 1;                       // last key any row of this wave sees
    const int kstride = n_heads * D;
    const T * kb = kmat + (size_t) e.kbase * kstride + h * D;
    const T * vb = vt + (size_t) h * D * ldv + e.kbase;
    constexpr int PER = PIECES / 256 > 0 ? PIECES / 256 : 1;
    bamd_u4 kr[PER], vr[PER];
    auto fetch = [&](int k0) {                                     // scratch rows are padded to whole 64s
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int c = tid + 256 * i;
            if (PIECES >= 256 || c < PIECES) {
                constexpr int pk = D * (int) sizeof(T) / 16, pv = 64 * (int) sizeof(T) / 16;
                kr[i] = *(const bamd_u4 *) ((const unsigned char *) (kb + (size_t) (k0 + c / pk) * kstride) + (c % pk) * 16);
                vr[i] = *(const bamd_u4 *) ((const unsigned char *) (vb + (size_t) (c / pv) * ldv + k0) + (c % pv) * 16);
            }
        }
    };
    fetch(0);
    for (int k0 = 0; k0 < len; k0 += 64) {
        __syncthreads();
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int c = tid + 256 * i;
            if (PIECES >= 256 || c < PIECES) {
                constexpr int pk = D * (int) sizeof(T) / 16, pv = 64 * (int) sizeof(T) / 16;
                *(bamd_u4 *) ((unsigned char *) (Ks + (c / pk) * KS) + (c % pk) * 16) = kr[i];
                *(bamd_u4 *) ((unsigned char *) (Vs + (c / pv) * VS) + (c % pv) * 16) = vr[i];
            }
        }
        __syncthreads();
        if (k0 + 64 < len) fetch(k0 + 64);
        if (k0 > w_hi || r0 >= e.n) continue;                      // nothing in this pass for this wave
        bamd_v4 sc[RT][4];
#pragma unroll
        for (int i = 0; i < RT; ++i)
#pragma unroll
            for (int t = 0; t < 4; ++t) sc[i][t] = bamd_v4{ 0, 0, 0, 0 };
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int k = 0; k < ND; ++k) {
                Frag<T> kf; kf.load(Ks + (t * 16 + lr) * KS + k * 32 + lq * 8);
#pragma unroll
                for (int i = 0; i < RT; ++i) sc[i][t] = mma(q[i][k], kf, sc[i][t]);
            }
        const bool all = k0 + 63 <= e.pos0 + r0;                   // every key of the pass is seen by every row
        float al[RT][4];
        bool moved = false;
#pragma unroll
        for (int i = 0; i < RT; ++i) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int pos = e.pos0 + r0 + i * 16 + lq * 4 + r;
                float mx = m[i][r];
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    float v = sc[i][t][r] * scale;
                    if (!all && k0 + t * 16 + lr > pos) v = -INFINITY;
                    mx = fmaxf(mx, v);
                }
                mx = row_max16(mx);
                al[i][r] = mx == -INFINITY ? 1.f : __builtin_amdgcn_exp2f(m[i][r] - mx);
                const float ref = mx == -INFINITY ? 0.f : mx;
                moved |= mx != m[i][r];
                float sum = 0.f;
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    float pe = __builtin_amdgcn_exp2f(fmaf(sc[i][t][r], scale, -ref));
                    if (!all && k0 + t * 16 + lr > pos) pe = 0.f;
                    sum += pe;
                    T * d = P + (i * 16 + lq * 4 + r) * VS + t * 16 + lr;
                    const T hi = to_act<T>(pe);
                    *d = hi;
                    if constexpr (NP == 2) d[16 * RT * VS] = to_act<T>(pe - (float) hi);
                }
                l[i][r] = l[i][r] * al[i][r] + sum; m[i][r] = mx;  // (sums of this lane's columns; added up at the end)
            }
        }
        if (__any(moved))                                          // (no maximum of the wave's rows has moved in most passes)
#pragma unroll
            for (int i = 0; i < RT; ++i)
#pragma unroll
                for (int j = 0; j < NV; ++j)
#pragma unroll
                    for (int r = 0; r < 4; ++r) o[i][j][r] *= al[i][r];
        wave_lds_fence();
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            Frag<T> pf[RT][NP];
#pragma unroll
            for (int i = 0; i < RT; ++i)
#pragma unroll
                for (int n = 0; n < NP; ++n) pf[i][n].load(P + (n * 16 * RT + i * 16 + lr) * VS + k * 32 + lq * 8);
#pragma unroll
            for (int j = 0; j < NV; ++j) {
                Frag<T> vf; vf.load(Vs + (j * 16 + lr) * VS + k * 32 + lq * 8);
#pragma unroll
                for (int i = 0; i < RT; ++i)
#pragma unroll
                    for (int n = 0; n < NP; ++n) o[i][j] = mma(pf[i][n], vf, o[i][j]);
            }
        }
        wave_lds_fence();
    }
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = r0 + i * 16 + lq * 4 + r;
            const float sum = row_sum16(l[i][r]);
            if (row >= e.n) continue;
            float f = 1.0f / sum;
            if (a.gated) f *= sigmoid_f(a.in[(size_t) (e.row0 + row) * a.ld + a.g_off + h]);
            const RowOut<Operand<T>> d = row_out<Operand<T>>(a.out, e.row0 + row, a.ldo, a.cb);
#pragma unroll
            for (int j = 0; j < NV; ++j) *d.at(h * D, j, lr) = to_operand<Operand<T>>(o[i][j][r] * f);
        }
}

// ---- decoding ---------------------------------------------------------------------------------------------------------------------------------------
// block (h * parts + part, row): q of head h carried into the latent space, four 16-row tiles of it; block (heads * parts, row): the row's own latent into the cache
template <typename T> __global__ void __launch_bounds__(256) latent_absorb_kernel(bamd_batch_dev b, bamd_latent_args a, T * qp, int parts) {
    __shared__ float red[16];
    __shared__ __align__(16) float q[256];
    const int h = blockIdx.x / parts, row = blockIdx.y;
    if (h == a.heads) { latent_store_row<T>(b, a, row, red); return; }
    const int lane = threadIdx.x & 63, kt_n = a.D / 32, rt_n = a.Rp / 16, hp = (a.heads + 15) / 16 * 16, rt = (blockIdx.x % parts) * 4 + (threadIdx.x >> 6);
    bamd_u4 w[8];
#pragma unroll
    for (int kt = 0; kt < 8; ++kt) w[kt] = rt < rt_n && kt < kt_n ? *(const bamd_u4 *) (a.ukT + ((((size_t) h * rt_n + rt) * kt_n + kt) * 64 + lane) * 8) : bamd_u4{ 0, 0, 0, 0 };
    for (int i = threadIdx.x; i < 256; i += 256) q[i] = i < a.D ? a.in[(size_t) row * a.ld + a.q_off + h * a.D + i] : 0.f;
    __syncthreads();
    float v = 0.f;
#pragma unroll
    for (int kt = 0; kt < 8; ++kt) {
        const float * x = q + kt * 32 + (lane >> 4) * 8;
        v += bf_lo(w[kt].x) * x[0] + bf_hi(w[kt].x) * x[1] + bf_lo(w[kt].y) * x[2] + bf_hi(w[kt].y) * x[3] + bf_lo(w[kt].z) * x[4] + bf_hi(w[kt].z) * x[5] + bf_lo(w[kt].w) * x[6] + bf_hi(w[kt].w) * x[7];
    }
    v += __shfl_xor(v, 16); v += __shfl_xor(v, 32);
    if (lane < 16 && rt < rt_n) qp[((size_t) row * hp + h) * a.Rp + rt * 16 + lane] = to_act<T>(v);
}
// block (split, head group of 16, row).  NR: 16-column tiles of the latent per wave; KEYS: keys per pass (64, or 32 where the rows are too wide for the LDS)
template <typename T, int NR, int KEYS>
__global__ void __launch_bounds__(256) latent_decode_kernel(bamd_batch_dev b, bamd_latent_args a, const T * qp, float * part_o, float * part_ml, int splits) {
    constexpr int PAD = 16 / sizeof(T), NP = sizeof(T) == 2 ? 2 : 1, PS = KEYS + PAD;
    constexpr int JM = NR * 64 * (int) sizeof(T) / 256, JB = JM < 1 ? 1 : JM > 4 ? 4 : JM;        // pieces of a row per thread, at once
    extern __shared__ __align__(16) unsigned char lds[];
    const int S = a.Rp + PAD;
    T * Cs = (T *) lds, * Qs = Cs + KEYS * S, * Ps = Qs + 16 * S;  // [KEYS][S], [16][S], [NP][16][PS]
    __shared__ float sc[16][KEYS + 1], mx[16], ls[16], al[16];
    const int sp = blockIdx.x, hg = blockIdx.y, row = blockIdx.z, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, lr = lane & 15, lq = lane >> 4;
    const bamd_entry e = b.ent[row];
    const int len = e.pos0 + 1, n_pg = (len + BAMD_PAGE - 1) / BAMD_PAGE, per = (n_pg + splits - 1) / splits, pg0 = sp * per, pg1 = min(n_pg, pg0 + per);
    const int hgs = gridDim.y, rt_n = a.Rp / 16, kt_n = a.Rp / 32, pr = a.Rp * (int) sizeof(T) / 16;
    if (tid < 16) { mx[tid] = -INFINITY; ls[tid] = 0.f; }
    const T * qsrc = qp + ((size_t) row * hgs * 16 + hg * 16) * a.Rp;
    for (int i = tid; i < 16 * pr; i += 256) *(bamd_u4 *) ((unsigned char *) (Qs + (i / pr) * S) + (i % pr) * 16) = *(const bamd_u4 *) ((const unsigned char *) qsrc + (size_t) i * 16);
    bamd_v4 o[NR];
#pragma unroll
    for (int j = 0; j < NR; ++j) o[j] = bamd_v4{ 0, 0, 0, 0 };
    for (int i = pg0 * (BAMD_PAGE / KEYS); i < pg1 * (BAMD_PAGE / KEYS); ++i) {
        const int pg = i / (BAMD_PAGE / KEYS), k0 = i * KEYS, n = min(KEYS, len - k0);      // keys k0 .. k0 + n - 1
        if (n <= 0) break;
        const unsigned char * src = (const unsigned char *) ((const T *) a.cache + (size_t) b.pages[(size_t) e.seq * b.max_pages + pg] * BAMD_PAGE * a.Rp + (size_t) (k0 % BAMD_PAGE) * a.Rp);
        __syncthreads();
        // sixteen threads per row, four rows per wave and load
        for (int j0 = 0; j0 < pr; j0 += 16 * JB) {
            bamd_u4 v[KEYS / 16][JB];
#pragma unroll
            for (int r4 = 0; r4 < KEYS / 16; ++r4)
#pragma unroll
                for (int j = 0; j < JB; ++j) { const int r = (tid >> 4) + 16 * r4, c = j0 + j * 16 + (tid & 15); v[r4][j] = r < n && c < pr ? *(const bamd_u4 *) (src + ((size_t) r * pr + c) * 16) : bamd_u4{ 0, 0, 0, 0 }; }
#pragma unroll
            for (int r4 = 0; r4 < KEYS / 16; ++r4)
#pragma unroll
                for (int j = 0; j < JB; ++j) { const int r = (tid >> 4) + 16 * r4, c = j0 + j * 16 + (tid & 15); if (c < pr) *(bamd_u4 *) ((unsigned char *) (Cs + r * S) + c * 16) = v[r4][j]; }
        }
        __syncthreads();
        if (wave * 16 < KEYS) {   // scores of 16 heads x this wave's 16 keys
            bamd_v4 s = { 0, 0, 0, 0 };
            for (int k = 0; k < kt_n; ++k) {
                Frag<T> qf, cf;
                qf.load(Qs + lr * S + k * 32 + lq * 8); cf.load(Cs + (wave * 16 + lr) * S + k * 32 + lq * 8);
                s = mma(qf, cf, s);
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) sc[lq * 4 + i][wave * 16 + lr] = wave * 16 + lr < n ? s[i] * a.scale : -INFINITY;
        }
        __syncthreads();
        {   // sixteen threads per head, KEYS / 16 keys each
            const int hd = tid >> 4, k = tid & 15;
            float v[KEYS / 16], m = mx[hd];
            const float m_old = m;
#pragma unroll
            for (int i = 0; i < KEYS / 16; ++i) { v[i] = sc[hd][k + 16 * i]; m = fmaxf(m, v[i]); }
            m = row_max16(m);
            float sum = 0.f;
#pragma unroll
            for (int i = 0; i < KEYS / 16; ++i) {
                const float p = __expf(v[i] - m);
                sum += p;
                const T hi = to_act<T>(p);
                Ps[hd * PS + k + 16 * i] = hi;
                if constexpr (NP == 2) Ps[(16 + hd) * PS + k + 16 * i] = to_act<T>(p - (float) hi);
            }
            sum = row_sum16(sum);
            if (k == 0) { const float f = __expf(m_old - m); al[hd] = f; ls[hd] = ls[hd] * f + sum; mx[hd] = m; }
        }
        __syncthreads();
        float f[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) f[i] = al[lq * 4 + i];
#pragma unroll
        for (int j = 0; j < NR; ++j)
#pragma unroll
            for (int i = 0; i < 4; ++i) o[j][i] *= f[i];
#pragma unroll
        for (int k = 0; k < KEYS / 32; ++k) {
            Frag<T> pf[NP];
#pragma unroll
            for (int n2 = 0; n2 < NP; ++n2) pf[n2].load(Ps + (n2 * 16 + lr) * PS + k * 32 + lq * 8);
#pragma unroll
            for (int j = 0; j < NR; ++j) {
                const int rt = wave + 4 * j;
                if (rt < rt_n) {
                    Frag<T> cf;
                    const T * c = Cs + (k * 32 + lq * 8) * S + rt * 16 + lr;
                    if constexpr (sizeof(T) == 2) {
#pragma unroll
                        for (int i = 0; i < 8; ++i) cf.v[i] = c[i * S];
                    } else {
#pragma unroll
                        for (int i = 0; i < 4; ++i) { cf.a[i] = c[i * S]; cf.b[i] = c[(i + 4) * S]; }
                    }
#pragma unroll
                    for (int n2 = 0; n2 < NP; ++n2) o[j] = mma(pf[n2], cf, o[j]);
                }
            }
        }
    }
    __syncthreads();
    const size_t base = ((size_t) row * hgs + hg) * splits + sp;
    float * po = part_o + base * 16 * a.Rp;
#pragma unroll
    for (int j = 0; j < NR; ++j) {
        const int rt = wave + 4 * j;
        if (rt < rt_n && pg0 < pg1)
#pragma unroll
            for (int i = 0; i < 4; ++i) po[(size_t) (lq * 4 + i) * a.Rp + rt * 16 + lr] = o[j][i];
    }
    if (tid < 16) { part_ml[(base * 16 + tid) * 2] = mx[tid]; part_ml[(base * 16 + tid) * 2 + 1] = ls[tid]; }
}
// block (head, row): the parts' sums, the sink, the value up-projection, the gate
template <typename T> __global__ void __launch_bounds__(512) latent_combine_kernel(bamd_batch_dev b, bamd_latent_args a, const float * __restrict__ part_o, const float * __restrict__ part_ml, int splits) {
    extern __shared__ __align__(16) float cl[];                    // [Rp] | part sums [groups][Rp]
    __shared__ float wsp[64];
    __shared__ float inv;
    const int h = blockIdx.x, row = blockIdx.y, hgs = (a.heads + 15) / 16, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, hh = h % 16;
    const int n_pg = (b.ent[row].pos0 + BAMD_PAGE) / BAMD_PAGE, per = (n_pg + splits - 1) / splits, live = (n_pg + per - 1) / per;      // parts that hold keys
    const size_t base = ((size_t) row * hgs + h / 16) * splits;
    if (wave == 0) {
        const float snk = a.sink ? a.sink[h] : -INFINITY;
        const float ms = lane < live ? part_ml[((base + lane) * 16 + hh) * 2] : -INFINITY, ls = lane < live ? part_ml[((base + lane) * 16 + hh) * 2 + 1] : 0.f;
        const float m = wave_max(fmaxf(snk, ms)), w = lane < live ? expf(ms - m) : 0.f;
        wsp[lane] = w;
        float sum = wave_sum(w * ls);
        if (a.sink) sum += expf(snk - m);
        if (lane == 0) inv = (a.gated ? sigmoid_f(a.in[(size_t) row * a.ld + a.g_off + h]) : 1.f) / sum;
    }
    __syncthreads();
    const int nq = a.Rp / 4, ng = 512 / nq, grp = tid / nq, q4 = (tid % nq) * 4;
    if (grp < ng) {
        bamd_v4 v = { 0, 0, 0, 0 };
        const float * src = part_o + (base * 16 + hh) * a.Rp + q4;
#pragma unroll 4
        for (int s = grp; s < live; s += ng) v = v + *(const bamd_v4 *) (src + (size_t) s * 16 * a.Rp) * wsp[s];
        *(bamd_v4 *) (cl + a.Rp * (1 + grp) + q4) = v;
    }
    __syncthreads();
    for (int r = tid; r < a.Rp; r += 512) {
        float v = 0.f;
#pragma unroll 8
        for (int g = 0; g < ng; ++g) v += cl[a.Rp * (1 + g) + r];
        cl[r] = v;
    }
    __syncthreads();
    const int kt_n = a.Rp / 32, vt_n = a.D / 16;
    for (int t = wave; t < vt_n; t += 8) {
        float v = 0.f;
        const bamd_u4 * wv = (const bamd_u4 *) (a.uv.w + (((size_t) h * vt_n + t) * kt_n * 64 + lane) * 8);
#pragma unroll 8
        for (int kt = 0; kt < kt_n; ++kt) {
            const bamd_u4 w = wv[(size_t) kt * 64];
            const float * x = cl + kt * 32 + (lane >> 4) * 8;
            v += bf_lo(w.x) * x[0] + bf_hi(w.x) * x[1] + bf_lo(w.y) * x[2] + bf_hi(w.y) * x[3] + bf_lo(w.z) * x[4] + bf_hi(w.z) * x[5] + bf_lo(w.w) * x[6] + bf_hi(w.w) * x[7];
        }
        v += __shfl_xor(v, 16); v += __shfl_xor(v, 32);
        if (lane < 16) *row_out<Operand<T>>(a.out, row, a.ldo, a.cb).at(h * a.D + t * 16 + lane) = to_operand<Operand<T>>(v * inv);
    }
}

// A decoded token of one head in one launch: block (head, row) of sixteen waves.  The query goes into the latent space (qp = W_uk^T q), the sequence's latents pass by in registers — a wave
// holds whole rows, takes their scores, and adds them up with their weights, all by itself — and the sixteen waves' sums, the token's own latent and the sink meet in front of the value
// up-projection.  The three launches above become one; the pass over the cache that sixteen heads share there is every head's own here, out of the L2.  W_uk and the first latents are requested
// before the token's row arrives.  Scores, weights and sums are 32-bit on the vector units: a head is one row of the matrix cores.
// KT: D / 32; NRT: sixteen-row tiles of W_uk per wave (Rp <= 256 NRT); NP: pieces of sixteen bytes of a latent per lane
// exp(x) of a share's maximum, x <= 0, to an ulp and a half.  __expf is off by half an ulp of x log2(e) (3e-6 at -62), and expf where products and sums may fuse is as well: its remainder enters twice
__device__ __forceinline__ float share_weight(float x) {
    const float hi = x * 1.4426950408889634f, lo = hi > -200.f ? fmaf(x, 1.9259629911266175e-8f, fmaf(x, 1.4426950408889634f, -hi)) : 0.f;
    return __builtin_amdgcn_exp2f(hi) * fmaf(lo, 0.6931471805599453f, 1.f);
}
template <typename T> __device__ __forceinline__ void piece_of(const bamd_u4 & w, float * x) {
    if constexpr (sizeof(T) == 2) { x[0] = bf_lo(w.x); x[1] = bf_hi(w.x); x[2] = bf_lo(w.y); x[3] = bf_hi(w.y); x[4] = bf_lo(w.z); x[5] = bf_hi(w.z); x[6] = bf_lo(w.w); x[7] = bf_hi(w.w); }
    else { x[0] = __uint_as_float(w.x); x[1] = __uint_as_float(w.y); x[2] = __uint_as_float(w.z); x[3] = __uint_as_float(w.w); }
}
template <typename T, int KT, int NRT, int NP> __global__ void __launch_bounds__(1024) latent_step_kernel(bamd_batch_dev b, bamd_latent_args a) {
    constexpr int VPP = 16 / (int) sizeof(T), D = 32 * KT, VT = D / 16, KP = 16 / VT, NKT = (8 * NRT + KP - 1) / KP, PF = NP == 2 ? 2 : NRT == 2 ? 3 : 4, RM = 256 * NRT;      // KP: shares of K per value tile
    extern __shared__ __align__(16) unsigned char lds[];
    __shared__ float q[D], qp[RM], own[RM], red[32], ms[257], ls[257], wt[257], part[16][16];
    const int h = blockIdx.x, row = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int rt_n = a.Rp / 16, kt_n = a.Rp / 32, pr = a.Rp / VPP;
    bamd_u4 wk[NRT][KT];
#pragma unroll
    for (int j = 0; j < NRT; ++j)
#pragma unroll
        for (int k = 0; k < KT; ++k) wk[j][k] = wave + 16 * j < rt_n ? *(const bamd_u4 *) (a.ukT + ((((size_t) h * rt_n + wave + 16 * j) * KT + k) * 64 + lane) * 8) : bamd_u4{ 0, 0, 0, 0 };
    const bamd_entry e = b.ent[row];
    const int past = e.pos0;
    const int32_t * const pages = b.pages + (size_t) e.seq * b.max_pages;
    const float * in = a.in + (size_t) row * a.ld;
    float qv = 0.f, cv = 0.f, cn = 0.f;
    static_assert(D <= 1024 && RM <= 1024, "a thread per value of the query and of the latent");
    if (tid < D) qv = in[a.q_off + h * D + tid];
    if (tid < a.R) { cv = in[a.c_off + tid]; cn = a.c_norm[tid]; }
    // rows of the cache: 2^lg lanes hold one (NP > 1: every lane NP pieces of one), a wave `rows` at a time, PF times in a batch; row (i * 16 + wave) * rows + lane >> lg.  A batch's rows never
    // straddle a page: `rows` is a power of two
    int lg = 0; while (lg < 6 && (1 << lg) < pr) ++lg;
    const int rows = 64 >> lg, sub = lane >> lg, px = lane & ((1 << lg) - 1);
    bamd_u4 pc[2][PF][NP];
    auto request = [&](int batch, auto to) {
#pragma unroll
        for (int i = 0; i < PF; ++i) {
            const int r0 = ((batch * PF + i) * 16 + wave) * rows, r = r0 + sub;
            const T * src = (const T *) a.cache + ((size_t) (r0 < past ? pages[r0 / BAMD_PAGE] : 0) * BAMD_PAGE + r % BAMD_PAGE) * a.Rp;
#pragma unroll
            for (int p = 0; p < NP; ++p) pc[decltype(to)::value][i][p] = r < past && px + 64 * p < pr ? *(const bamd_u4 *) (src + (px + 64 * p) * VPP) : bamd_u4{ 0, 0, 0, 0 };
        }
    };
    const int batches = (past + PF * 16 * rows - 1) / (PF * 16 * rows);
    const std::integral_constant<int, 0> even; const std::integral_constant<int, 1> odd;
    request(0, even); request(1, odd);
    float sq[1] = { cv * cv };
    if (tid < D) q[tid] = qv;
    block_sum<1>(sq, red);                                         // (its barriers publish q as well)
    if (tid < a.Rp) {                                              // as it is cached
        const T v = to_act<T>(tid < a.R ? cv * (1.0f / sqrtf(sq[0] / (float) a.R + a.eps)) * cn : 0.f);
        own[tid] = (float) v;
        if (h == 0) ((T *) a.cache)[((size_t) pages[past / BAMD_PAGE] * BAMD_PAGE + past % BAMD_PAGE) * a.Rp + tid] = v;
    }
#pragma unroll
    for (int j = 0; j < NRT; ++j) {
        float v = 0.f;
#pragma unroll
        for (int k = 0; k < KT; ++k) {
            const float * x = q + k * 32 + (lane >> 4) * 8;
            const bamd_u4 w = wk[j][k];
            v += bf_lo(w.x) * x[0] + bf_hi(w.x) * x[1] + bf_lo(w.y) * x[2] + bf_hi(w.y) * x[3] + bf_lo(w.z) * x[4] + bf_hi(w.z) * x[5] + bf_lo(w.w) * x[6] + bf_hi(w.w) * x[7];
        }
        v += __shfl_xor(v, 16); v += __shfl_xor(v, 32);
        if (lane < 16 && wave + 16 * j < rt_n) qp[(wave + 16 * j) * 16 + lane] = v;
    }
    bamd_u4 wv[NKT];                                               // of this wave's value tile and share of K
    const int vt = wave % VT, kp = wave / VT;
#pragma unroll
    for (int k = 0; k < NKT; ++k) wv[k] = k * KP + kp < kt_n ? *(const bamd_u4 *) (a.uv.w + ((((size_t) h * VT + vt) * kt_n + k * KP + kp) * 64 + lane) * 8) : bamd_u4{ 0, 0, 0, 0 };
    __syncthreads();
    float qx[NP][VPP], o[NP][VPP], m = -INFINITY, l = 0.f;
#pragma unroll
    for (int p = 0; p < NP; ++p)
#pragma unroll
        for (int i = 0; i < VPP; ++i) { qx[p][i] = px + 64 * p < pr ? qp[(px + 64 * p) * VPP + i] : 0.f; o[p][i] = 0.f; }
    auto take = [&](int batch, auto from) {
        float s[PF], mx = m;
#pragma unroll
        for (int i = 0; i < PF; ++i) {
            float v = 0.f;
#pragma unroll
            for (int p = 0; p < NP; ++p) {
                float x[VPP];
                piece_of<T>(pc[decltype(from)::value][i][p], x);
#pragma unroll
                for (int k = 0; k < VPP; ++k) v += qx[p][k] * x[k];
            }
            s[i] = v;
        }
        if (lg >= 4) {
#pragma unroll
            for (int i = 0; i < PF; ++i) s[i] = row_sum16(s[i]);
        } else for (int d = 1; d < (1 << lg); d *= 2)
#pragma unroll
            for (int i = 0; i < PF; ++i) s[i] += __shfl_xor(s[i], d);
        if (lg >= 5)
#pragma unroll
            for (int i = 0; i < PF; ++i) s[i] += __shfl_xor(s[i], 16);
        if (lg >= 6)
#pragma unroll
            for (int i = 0; i < PF; ++i) s[i] += __shfl_xor(s[i], 32);
#pragma unroll
        for (int i = 0; i < PF; ++i) { s[i] = ((batch * PF + i) * 16 + wave) * rows + sub < past ? s[i] * a.scale : -INFINITY; mx = fmaxf(mx, s[i]); }
        const float ref = mx == -INFINITY ? 0.f : mx, f = __expf(m - ref);          // (no rows yet: nothing to rescale)
        l *= f; m = mx;
#pragma unroll
        for (int p = 0; p < NP; ++p)
#pragma unroll
            for (int k = 0; k < VPP; ++k) o[p][k] *= f;
#pragma unroll
        for (int i = 0; i < PF; ++i) {
            const float w = __expf(s[i] - ref);
            l += w;
#pragma unroll
            for (int p = 0; p < NP; ++p) {
                float x[VPP];
                piece_of<T>(pc[decltype(from)::value][i][p], x);
#pragma unroll
                for (int k = 0; k < VPP; ++k) o[p][k] += w * x[k];
            }
        }
    };
    for (int t = 0; t < batches; t += 2) {
        take(t, even); request(t + 2, even);
        if (t + 1 < batches) { take(t + 1, odd); request(t + 3, odd); }
    }
    // sixteen waves x `rows` sums, the own latent behind them
    float * const ps = (float *) lds;                              // [16 rows][Rp]
    const int n = 16 * rows, at = wave * rows + sub;
#pragma unroll
    for (int p = 0; p < NP; ++p)
        if (px + 64 * p < pr)
#pragma unroll
            for (int k = 0; k < VPP; ++k) ps[at * a.Rp + (px + 64 * p) * VPP + k] = o[p][k];
    if (px == 0) { ms[at] = m; ls[at] = l; }
    if (wave == 0) {
        float v = 0.f;
        for (int r = lane; r < a.Rp; r += 64) v += qp[r] * own[r];
        v = wave_sum(v) * a.scale;
        if (lane == 0) { ms[n] = v; ls[n] = 1.f; }
    }
    __syncthreads();
    const float snk = a.sink ? a.sink[h] : -INFINITY;
    float mx = fmaxf(snk, ms[n]);
    for (int i = lane; i < n; i += 64) mx = fmaxf(mx, ms[i]);
    mx = wave_max(mx);
    if (tid <= n) wt[tid] = share_weight(ms[tid] - mx);
    __syncthreads();
    float sum = 0.f;
    for (int i = lane; i <= n; i += 64) sum += wt[i] * ls[i];
    sum = wave_sum(sum);
    if (a.sink) sum += expf(snk - mx);
    const int th = a.Rp <= 256 ? 4 : 2, r = tid / th, g = tid % th;          // th threads per value of the latent: neighbours
    float v = 0.f;
    if (r < a.Rp) {
        for (int i = g; i < n; i += th) v += wt[i] * ps[i * a.Rp + r];
        if (g == 0) v += wt[n] * own[r];
    }
    v += __shfl_xor(v, 1); if (th == 4) v += __shfl_xor(v, 2);
    if (r < a.Rp && g == 0) qp[r] = v;                             // (the scores are behind a barrier)
    __syncthreads();
    v = 0.f;
#pragma unroll
    for (int k = 0; k < NKT; ++k)
        if (k * KP + kp < kt_n) {
            const float * x = qp + (k * KP + kp) * 32 + (lane >> 4) * 8;
            const bamd_u4 w = wv[k];
            v += bf_lo(w.x) * x[0] + bf_hi(w.x) * x[1] + bf_lo(w.y) * x[2] + bf_hi(w.y) * x[3] + bf_lo(w.z) * x[4] + bf_hi(w.z) * x[5] + bf_lo(w.w) * x[6] + bf_hi(w.w) * x[7];
        }
    v += __shfl_xor(v, 16); v += __shfl_xor(v, 32);
    if (lane < 16) part[wave][lane] = v;
    __syncthreads();
    if (tid >= D) return;
    v = 0.f;
#pragma unroll
    for (int k = 0; k < KP; ++k) v += part[k * VT + tid / 16][tid % 16];
    *row_out<Operand<T>>(a.out, row, a.ldo, a.cb).at(h * D + tid) = to_operand<Operand<T>>(v * ((a.gated ? sigmoid_f(in[a.g_off + h]) : 1.f) / sum));
}

// ---- launches ---------------------------------------------------------------------------------------------------------------------------------------
void bamd_launch_latent_store(int act, const bamd_batch_dev & b, const bamd_latent_args & a, hipStream_t s) {
    if (act == BAMD_ACT_F32) hipLaunchKernelGGL(latent_store_kernel<float>, dim3(b.rows), dim3(256), 0, s, b, a);
    else hipLaunchKernelGGL(latent_store_kernel<bamd_bf>, dim3(b.rows), dim3(256), 0, s, b, a);
}
void bamd_launch_latent_gather(int act, const bamd_batch_dev & b, const bamd_latent_args & a, const int32_t * k_entry, int k_rows, void * dst, hipStream_t s) {
    if (act == BAMD_ACT_F32) hipLaunchKernelGGL(latent_gather_kernel<float>, dim3(k_rows / BAMD_PAGE), dim3(256), 0, s, b, a, k_entry, (float *) dst);
    else hipLaunchKernelGGL(latent_gather_kernel<bamd_bf>, dim3(k_rows / BAMD_PAGE), dim3(256), 0, s, b, a, k_entry, (bamd_bf *) dst);
}
static int prompt_rt(int act, int D) { return act == BAMD_ACT_F32 ? 1 : D <= 128 ? 2 : 1; }
int bamd_latent_prompt_rows(int act, int D) { return 64 * prompt_rt(act, D); }
template <typename T, int ND, int RT>
static void prompt_go(const bamd_batch_dev & b, const bamd_latent_args & a, const bamd_qtile * tiles, int n, const void * k, const void * vt, int ldv, hipStream_t s) {
    constexpr int D = ND * 32, KS = D + 16 / sizeof(T), VS = 64 + 16 / sizeof(T), NP = sizeof(T) == 2 ? 2 : 1;
    const size_t lds = sizeof(T) * ((size_t) 64 * KS + (size_t) D * VS + (size_t) 4 * NP * 16 * RT * VS);
    hipLaunchKernelGGL((latent_prompt_kernel<T, ND, RT>), dim3(n * a.heads), dim3(256), lds, s, b, a, tiles, a.heads, (const T *) k, (const T *) vt, ldv);
}
int bamd_launch_latent_prompt(int act, const bamd_batch_dev & b, const bamd_latent_args & a, const bamd_qtile * tiles, int n, const void * k, const void * vt, int ldv, hipStream_t s) {
    if (n < 1 || (ldv & 63)) return 1;
    if (act == BAMD_ACT_F32) switch (a.D) {
        case 32: prompt_go<float, 1, 1>(b, a, tiles, n, k, vt, ldv, s); return 0;
        case 64: prompt_go<float, 2, 1>(b, a, tiles, n, k, vt, ldv, s); return 0;
        case 128: prompt_go<float, 4, 1>(b, a, tiles, n, k, vt, ldv, s); return 0;
        case 256: prompt_go<float, 8, 1>(b, a, tiles, n, k, vt, ldv, s); return 0;
    } else switch (a.D) {
        case 32: prompt_go<bamd_bf, 1, 2>(b, a, tiles, n, k, vt, ldv, s); return 0;
        case 64: prompt_go<bamd_bf, 2, 2>(b, a, tiles, n, k, vt, ldv, s); return 0;
        case 128: prompt_go<bamd_bf, 4, 2>(b, a, tiles, n, k, vt, ldv, s); return 0;
        case 256: prompt_go<bamd_bf, 8, 1>(b, a, tiles, n, k, vt, ldv, s); return 0;
    }
    return 1;
}
template <typename T> static size_t decode_lds(int Rp, int keys) { return sizeof(T) * ((size_t) (keys + 16) * (Rp + 16 / sizeof(T)) + 2 * 16 * (keys + 16 / sizeof(T))); }
#define DECODE_LDS (152 * 1024)
int bamd_latent_max_rank(int act) {                                // widest latent row with a decoding kernel
    int rp = 1024;
    while ((act == BAMD_ACT_F32 ? decode_lds<float>(rp, 32) : decode_lds<bamd_bf>(rp, 32)) > DECODE_LDS) rp -= 32;
    return rp;
}
template <typename T, int KEYS>
static void decode_pick(const bamd_batch_dev & b, const bamd_latent_args & a, const T * qp, float * po, float * pm, int splits, hipStream_t s) {
    const dim3 grid(splits, (a.heads + 15) / 16, b.rows);
    const size_t lds = decode_lds<T>(a.Rp, KEYS);
    const int nr = (a.Rp / 16 + 3) / 4;
    if (nr <= 1) hipLaunchKernelGGL((latent_decode_kernel<T, 1, KEYS>), grid, dim3(256), lds, s, b, a, qp, po, pm, splits);
    else if (nr <= 2) hipLaunchKernelGGL((latent_decode_kernel<T, 2, KEYS>), grid, dim3(256), lds, s, b, a, qp, po, pm, splits);
    else if (nr <= 4) hipLaunchKernelGGL((latent_decode_kernel<T, 4, KEYS>), grid, dim3(256), lds, s, b, a, qp, po, pm, splits);
    else if (nr <= 8) hipLaunchKernelGGL((latent_decode_kernel<T, 8, KEYS>), grid, dim3(256), lds, s, b, a, qp, po, pm, splits);
    else hipLaunchKernelGGL((latent_decode_kernel<T, 16, KEYS>), grid, dim3(256), lds, s, b, a, qp, po, pm, splits);
}
template <typename T>
static int decode_go(const bamd_batch_dev & b, const bamd_latent_args & a, void * qp, float * part_o, float * part_ml, int splits, hipStream_t s) {
    if (splits < 1 || splits > 64 || a.Rp > 1024 || decode_lds<T>(a.Rp, 32) > DECODE_LDS) return 1;
    const int parts = (a.Rp / 16 + 3) / 4;
    hipLaunchKernelGGL(latent_absorb_kernel<T>, dim3(a.heads * parts + 1, b.rows), dim3(256), 0, s, b, a, (T *) qp, parts);
    if (decode_lds<T>(a.Rp, 64) <= DECODE_LDS) decode_pick<T, 64>(b, a, (const T *) qp, part_o, part_ml, splits, s);
    else decode_pick<T, 32>(b, a, (const T *) qp, part_o, part_ml, splits, s);
    hipLaunchKernelGGL(latent_combine_kernel<T>, dim3(a.heads, b.rows), dim3(512), ((size_t) a.Rp + 2048) * 4, s, b, a, part_o, part_ml, splits);
    return 0;
}
template <typename T, int KT> static void step_pick(const bamd_batch_dev & b, const bamd_latent_args & a, hipStream_t s) {
    constexpr int VPP = 16 / (int) sizeof(T);
    int lanes = 1; while (lanes < 64 && lanes < a.Rp / VPP) lanes *= 2;
    const size_t lds = (size_t) 16 * (64 / lanes) * a.Rp * 4;
    const dim3 grid(a.heads, b.rows);
    if (a.Rp <= 256) hipLaunchKernelGGL((latent_step_kernel<T, KT, 1, 1>), grid, dim3(1024), lds, s, b, a);
    else hipLaunchKernelGGL((latent_step_kernel<T, KT, 2, 16 / VPP / 2>), grid, dim3(1024), lds, s, b, a);
}
template <typename T> static void step_go(const bamd_batch_dev & b, const bamd_latent_args & a, hipStream_t s) {
    if (a.D == 32) step_pick<T, 1>(b, a, s); else if (a.D == 64) step_pick<T, 2>(b, a, s); else step_pick<T, 4>(b, a, s);
}
bool bamd_latent_step_valid(int D, int Rp) { return D <= 128 && Rp <= 512; }
// Every head reads the cache by itself in the one launch, sixteen share it in the three: 20 to 25 us less a step against a time per position that goes by the rank and 42 numbers (a row's sum over its lanes
// and its weight cost the same whatever it holds): where both are level, positions x (rank + 42) are 180k to 210k at ranks 32 to 512 in bfloat16 and 140k to 170k in 32-bit.  Steps of eight layers, three
// launches and one, us: width 2048, rank 256, 16 heads: 60 positions 423 | 398, 155 427 | 408, 380 428 | 418, 800 432 | 438; sixteen rows 216 709 | 689, 500 707 | 692, 1000 711 | 716; 32-bit 155
// 461 | 430, 380 460 | 452, 800 461 | 501.  Width 4096, rank 512, 32 heads: 155 830 | 809, 380 838 | 836, 800 827 | 884; sixteen rows 216 1280 | 1253, 500 1289 | 1317; 32-bit 155 907 | 849.
// Lower ranks: width 1024, 8 heads, rank 32 2000 positions 267 | 261, 3000 266 | 267, 4000 264 | 273; 64 1500 265 | 261, 2000 266 | 268, 3000 266 | 280; 128 1000 277 | 271, 1500 279 | 284, 2000 280 | 297; 16
// heads of width 2048, rank 64 1000 378 | 366, 2000 381 | 384, six rows 489 | 483, rank 256 520 392 | 384, 640 385 | 391; 32-bit rank 32 1700 272 | 268, 3000 276 | 284; 64 1000 274 | 265, 1700 277 | 281; 128 500 290 | 267, 1000 284 | 285; 256 430 415 | 406.
// With more than two blocks to a CU the three are ahead: 48 rows of 16 heads, 100 positions 1200 | 1223
bool bamd_latent_one_launch(int act, int D, int Rp, int rows, int heads, int most) {
    return bamd_latent_step_valid(D, Rp) && most > 0 && (size_t) most * (Rp + 42) <= (act == BAMD_ACT_F32 ? 140000 : 180000) && rows * heads <= 512;
}
void bamd_launch_latent_step(int act, const bamd_batch_dev & b, const bamd_latent_args & a, hipStream_t s) {
    if (act == BAMD_ACT_F32) step_go<float>(b, a, s); else step_go<bamd_bf>(b, a, s);
}
int bamd_launch_latent_decode(int act, const bamd_batch_dev & b, const bamd_latent_args & a, void * qp, float * part_o, float * part_ml, int splits, hipStream_t s) {
    return act == BAMD_ACT_F32 ? decode_go<float>(b, a, qp, part_o, part_ml, splits, s) : decode_go<bamd_bf>(b, a, qp, part_o, part_ml, splits, s);
}
