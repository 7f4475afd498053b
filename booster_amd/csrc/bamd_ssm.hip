// bamd_ssm.hip — the state-space recurrence (Mamba-2 form): S_t = exp(-exp(A_log) dt_t) S_(t-1) + dt_t B_t x_t^T, y_t = S_t^T C_t + D x_t, gated by silu(z_t).
//
//   prompts: ssm_conv_kernel filters x, B and C and computes step sizes and decays for all tokens, ssm_chunk_kernel takes them sixteen at a time on the f32 matrix cores;
//   decoding (one token): ssm_step_kernel, a block per (PT value columns, head, sequence), filters its own channels, one launch in all.  A lane keeps four columns of NPL state
//     rows in registers (lane = column quad + group of state rows, so that a row's B and C serve four columns from one LDS read); y is summed over a lane's rows, then over the groups.
// The state is read and written once per step; everything is 32-bit.
#include <algorithm>
#include "bamd_dense_device.h"
#include <type_traits>

struct SsmIndex {                                                  // channels of one (column block, head): [x columns | B | C]
    int h, g, p0, pw, inner, ch, N, groups, P;
    __device__ __forceinline__ int channel(int c) const { return c < pw ? h * P + p0 + c : c < pw + N ? inner + g * N + (c - pw) : inner + (groups + g) * N + (c - pw - N); }
};
// input of channel q at place t of the step (negative: before it)
__device__ __forceinline__ float ssm_raw(const bamd_ssm_args & a, const float * in, const float * hist, int t, int q, int inner, int ch) {
    return t >= 0 ? in[(size_t) t * a.ld + inner + q] : hist ? hist[(size_t) (a.taps - 1 + t) * ch + q] : 0.f;
}
__device__ __forceinline__ float ssm_filter(const bamd_ssm_args & a, const float * in, const float * hist, int t, int q, int inner, int ch) {
    float v = a.conv_b[q];
    for (int k = 0; k < a.taps; ++k) v = fmaf(a.conv[(size_t) q * a.taps + k], ssm_raw(a, in, hist, t - (a.taps - 1) + k, q, inner, ch), v);
    return silu_f(v);
}

// prompts: filtered [rows][ch] and {dt, decay} [rows][heads]; block (256 channels, SSM_STRIP rows).  FOUR: four taps, their inputs kept in registers from row to row.  The
// block of a sequence's last row also stores the convolutions' last inputs
#define SSM_STRIP 8
template <bool FOUR>
__global__ void __launch_bounds__(256) ssm_conv_kernel(bamd_batch_dev b, bamd_ssm_args a) {
    const int inner = a.heads * a.P, ch = inner + 2 * a.groups * a.N, q = blockIdx.x * 256 + threadIdx.x, T1 = a.taps - 1;
    const int row0 = blockIdx.y * SSM_STRIP, row1 = min(row0 + SSM_STRIP, b.rows);
    float w[4] = { 0, 0, 0, 0 }, x[4] = { 0, 0, 0, 0 }, bias = 0.f, eA = 0.f, dtb = 0.f;
    if (FOUR && q < ch) {
#pragma unroll
        for (int k = 0; k < 4; ++k) w[k] = a.conv[(size_t) q * 4 + k];
        bias = a.conv_b[q];
    }
    if (q < a.heads) { eA = expf(a.A_log[q]); dtb = a.dt_bias[q]; }
    int at = -1;
    bamd_entry e = {};
    for (int row = row0; row < row1; ++row) {
        const int i = b.row_entry[row];
        const bool fresh = i != at;
        if (fresh) { e = b.ent[i]; at = i; }
        const int t = row - e.row0;
        const float * in = a.in + (size_t) e.row0 * a.ld;
        const float * hist = e.pos0 > 0 ? a.hist + ((size_t) e.par * b.n_seq + e.seq) * T1 * ch : nullptr;
        if (q < ch) {
            float v;
            if (FOUR) {
                if (fresh) for (int k = 1; k < 4; ++k) x[k] = ssm_raw(a, in, hist, t - 4 + k, q, inner, ch);
                x[0] = x[1]; x[1] = x[2]; x[2] = x[3]; x[3] = in[(size_t) t * a.ld + inner + q];
                v = bias;
#pragma unroll
                for (int k = 0; k < 4; ++k) v = fmaf(w[k], x[k], v);
                v = silu_f(v);
            } else v = ssm_filter(a, in, hist, t, q, inner, ch);
            a.filtered[(size_t) row * ch + q] = v;
            if (t == e.n - 1) {
                float * ho = a.hist + ((size_t) (e.par ^ 1) * b.n_seq + e.seq) * T1 * ch;
                for (int r = 0; r < T1; ++r) ho[(size_t) r * ch + q] = ssm_raw(a, in, hist, e.n - T1 + r, q, inner, ch);
            }
        }
        if (q < a.heads) {
            const float dt = softplus_f(in[(size_t) t * a.ld + inner + ch + q] + dtb);
            a.steps[((size_t) row * a.heads + q) * 2] = dt; a.steps[((size_t) row * a.heads + q) * 2 + 1] = expf(-eA * dt);
        }
    }
}

// Decoding, one token.  PT columns per block (16, 32, 64); NPL state rows per lane; 4 * (256 / PT) row groups over the four waves.  FOUR: four taps.
// What bounds a block is its chain of reads: everything is asked for before anything is waited for, the inputs of the filters first (a loop over the taps, each of its reads waited for, and the
// inputs read again for the next step's history: 64 heads x 64 x 128 took 8.2 us, now 5.8)
template <int PT, int NPL, bool FOUR>
__global__ void __launch_bounds__(256) ssm_step_kernel(bamd_batch_dev b, bamd_ssm_args a) {
    constexpr int Q = PT / 4, NG = 64 / Q, GROUPS = 4 * NG, NP = GROUPS * NPL;     // NP >= N state rows
    __shared__ __align__(16) float ops[PT + 2 * NP], yp[GROUPS][PT];
    float * xs = ops, * Bs = ops + PT, * Cs = ops + PT + NP;
    __shared__ float sdt, sdec;
    const bamd_entry e = b.ent[blockIdx.z];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, quad = lane % Q, grp = wave * NG + lane / Q;
    SsmIndex ix;
    ix.h = blockIdx.y; ix.p0 = blockIdx.x * PT; ix.pw = min(PT, a.P - ix.p0); ix.N = a.N; ix.groups = a.groups; ix.P = a.P; ix.inner = a.heads * a.P; ix.ch = ix.inner + 2 * a.groups * a.N;
    const int per = a.heads / a.groups, N = a.N, T1 = a.taps - 1, CH = ix.pw + 2 * N;
    ix.g = ix.h / per;
    const float * in = a.in + (size_t) e.row0 * a.ld;
    float * st = a.state + (((size_t) e.seq * a.heads + ix.h) * N) * a.P + ix.p0;
    const float * hist = e.pos0 > 0 ? a.hist + ((size_t) e.par * b.n_seq + e.seq) * T1 * ix.ch : nullptr;
    constexpr int CF = (PT + 2 * NP + 255) / 256;                  // channels per thread
    float x[CF][4], cw[CF][4], cb[CF];
    if constexpr (FOUR)
#pragma unroll
        for (int f = 0; f < CF; ++f) {
            const int q = ix.channel(min(tid + 256 * f, CH - 1));
#pragma unroll
            for (int k = 0; k < 3; ++k) x[f][k] = hist ? hist[(size_t) k * ix.ch + q] : 0.f;
            x[f][3] = in[ix.inner + q]; cb[f] = a.conv_b[q];
#pragma unroll
            for (int k = 0; k < 4; ++k) cw[f][k] = a.conv[(size_t) q * 4 + k];
        }
    const float dt_in = in[ix.inner + ix.ch + ix.h], dt_b = a.dt_bias[ix.h], A_log = a.A_log[ix.h], D = a.D[ix.h], gate = in[ix.h * a.P + ix.p0 + min(tid, ix.pw - 1)];
    // sixteen bytes at a time where rows start on sixteen bytes (pw is then a multiple of four as well), from a place clamped into the state: a branch around each of 4 NPL single values
    // made sixteen sequences of 128 heads x 64 x 128 take 48 us for 134 MB, now 31
    const bool wide = (a.P & 3) == 0;
    bamd_v4 s[NPL];
    if (wide) {
#pragma unroll
        for (int j = 0; j < NPL; ++j) s[j] = *(const bamd_v4 *) (st + (size_t) min(grp * NPL + j, N - 1) * a.P + min(quad * 4, ix.pw - 4));
#pragma unroll
        for (int j = 0; j < NPL; ++j) if (!(e.pos0 > 0 && grp * NPL + j < N && quad * 4 < ix.pw)) s[j] = bamd_v4{ 0, 0, 0, 0 };
    } else {
#pragma unroll
        for (int j = 0; j < NPL; ++j)
#pragma unroll
            for (int k = 0; k < 4; ++k) { const int n = grp * NPL + j, p = quad * 4 + k; s[j][k] = (e.pos0 > 0 && n < N && p < ix.pw) ? st[(size_t) n * a.P + p] : 0.f; }
    }
    for (int i = tid; i < PT + 2 * NP; i += 256) ops[i] = 0.f;
    auto slot = [&](int c) { return c < ix.pw ? c : c < ix.pw + N ? PT + (c - ix.pw) : PT + NP + (c - ix.pw - N); };
    __syncthreads();                                               // zeroes are in
    float * ho = a.hist + ((size_t) (e.par ^ 1) * b.n_seq + e.seq) * T1 * ix.ch;
    const int own = (ix.h % per == 0 && ix.p0 == 0) ? CH : ix.pw;     // B and C belong to the group: its first head's first block stores their inputs
    if constexpr (FOUR) {
#pragma unroll
        for (int f = 0; f < CF; ++f) {
            const int c = tid + 256 * f;
            if (c >= CH) continue;
            float v = cb[f];
#pragma unroll
            for (int k = 0; k < 4; ++k) v = fmaf(cw[f][k], x[f][k], v);
            ops[slot(c)] = silu_f(v);
            if (c < own)
#pragma unroll
                for (int r = 0; r < 3; ++r) ho[(size_t) r * ix.ch + ix.channel(c)] = x[f][r + 1];
        }
    } else for (int c = tid; c < CH; c += 256) {
        const int q = ix.channel(c);
        ops[slot(c)] = ssm_filter(a, in, hist, 0, q, ix.inner, ix.ch);
        if (c < own) for (int r = 0; r < T1; ++r) ho[(size_t) r * ix.ch + q] = ssm_raw(a, in, hist, 1 - T1 + r, q, ix.inner, ix.ch);
    }
    if (tid == 255) { const float dt = softplus_f(dt_in + dt_b); sdt = dt; sdec = expf(-expf(A_log) * dt); }
    __syncthreads();
    {
        const float d = sdec, dt = sdt;
        const bamd_v4 x4 = *(const bamd_v4 *) &xs[quad * 4];
        float xv[4], y[4] = { 0.f, 0.f, 0.f, 0.f };
#pragma unroll
        for (int k = 0; k < 4; ++k) xv[k] = dt * x4[k];
#pragma unroll
        for (int j = 0; j < NPL; ++j) {
            const float B = Bs[grp * NPL + j], C = Cs[grp * NPL + j];
#pragma unroll
            for (int k = 0; k < 4; ++k) { s[j][k] = fmaf(d, s[j][k], B * xv[k]); y[k] = fmaf(C, s[j][k], y[k]); }
        }
        *(bamd_v4 *) &yp[grp][quad * 4] = bamd_v4{ y[0], y[1], y[2], y[3] };
    }
    __syncthreads();
    if (tid < ix.pw) {
        float y[4] = { 0.f, 0.f, 0.f, 0.f };
#pragma unroll
        for (int g = 0; g < GROUPS; ++g) y[g & 3] += yp[g][tid];
        a.out[(size_t) e.row0 * a.ldo + ix.h * a.P + ix.p0 + tid] = ((y[0] + y[1]) + (y[2] + y[3]) + D * xs[tid]) * silu_f(gate);
    }
    if (wide) {
#pragma unroll
        for (int j = 0; j < NPL; ++j) if (grp * NPL + j < N && quad * 4 < ix.pw) *(bamd_v4 *) (st + (size_t) (grp * NPL + j) * a.P + quad * 4) = s[j];
        return;
    }
#pragma unroll
    for (int j = 0; j < NPL; ++j)
#pragma unroll
        for (int k = 0; k < 4; ++k) { const int n = grp * NPL + j, p = quad * 4 + k; if (n < N && p < ix.pw) st[(size_t) n * a.P + p] = s[j][k]; }
}

// Prompts: the tokens of a sequence sixteen at a time on the f32 matrix cores.  With p_t the product of the decays up to t inside a chunk and f_s that of the decays behind s,
//     y_t = p_t C_t^T S + sum over s <= t of (C_t . B_s) (product of the decays s + 1 .. t) dt_s x_s,     S <- p_15 S + sum over s of B_s (f_s dt_s x_s)^T;
// every factor is a product of at most sixteen decays, nothing is divided or taken from a difference of sums.  A block is 32 value columns of a head: eight waves, two tiles of 16
// columns x four quarters of the state rows (y is summed over the quarters); a wave keeps its NT 16 x 16 tiles of S as accumulators, which are at once the operand that C^T S needs
// (the four rows a lane holds are the four steps of a 16x16x4 product), as B^T C comes out in the order that its product with x wants.  Chunk c + 2 is requested and chunk c + 1 put
// into LDS while c is computed.  One token after the other on the vector ALUs was a chain of 283 ns per token: 2048 tokens of 128 heads x 64 x 128 took 525 us; now 271.  A chunk's
// matrix instructions take 0.4 us of a SIMD's time; the rest is what stands between them, which is why two waves share a SIMD (four waves a block: 331 us).
// The products meet a later token's B, C and x with a factor of zero, which hides any finite value; an infinity, a NaN or a product that overflows shows as a y that is not finite.  Then the
// wave takes the chunk again one token after the other, from the state in front of it, so that such a token reaches those behind it and none in front.  (A look at every value on
// its way into LDS instead cost 264 us for 258; this one, under the stores of y, nothing.)
// A prompt of few heads leaves CUs idle, and tokens one behind the other are its time: up to four parts of its tokens are taken at once, each by a block of its own, which brings the state along from the
// first token on without the outputs (half a chunk's time).  Where values stay finite these are the bits that one block gets.  A chunk that one block takes again for its outputs (a C that is not finite) is
// not taken again by those that bring only the state along: what stays finite behind it may be rounded otherwise, by the number of parts.  Borders are where all parts end together.  Four layers, us, one part and those taken: width 2048
// (64 heads, two parts) 131 tokens 573 | 567, 1000 1228 | 1164, 2048 2051 | 1907; 1024 (32 heads, four) 300 473 | 448, 2048 1410 | 1217; 600 (13 heads) 1000 723 | 621.  Two parts to a CU (128 heads) were
// no faster (2048 tokens of width 4096 4268 | 4271).  All these are state 128.  Tokens in one part have an instance of their own: with the parts' code in it a state of up to 64 takes 130 registers for
// 128, one block per CU for two.  Eight prompts of 330 to 186 tokens, width 2048, state 64, 2320 us with, 2231 without, state 32 2312 | 2220; width 4096 (128 heads), two prompts of 900 and 675 3804 | 3700
#define SSM_AGAIN 0.55f                             /* a chunk whose outputs are taken costs 1, one that only brings the state along 1 - this */
struct ssm_cut { float at[3]; };                   // inner borders, of all tokens
template <int NT, bool PARTS>
__global__ void __launch_bounds__(512) ssm_chunk_kernel(bamd_batch_dev b, bamd_ssm_args a, int cols, ssm_cut cut) {
    constexpr int NQ = 4, NP = 16 * NQ * NT, LB = NP + 4, LX = 36, LD = 20, PF = 16 * NP / 512, KS = 512 / NP;      // row lengths in LDS: four rows on, 16 banks on
    __shared__ __align__(16) float Bs[2][16 * LB], Cs[2][16 * LB], xs[2][16 * LX], yp[2][NQ][16 * LX], dm[2][16 * LD];
    __shared__ __align__(16) float pre[2][16], fd[2][16], dts[2][16];
    const bamd_entry e = b.ent[blockIdx.z];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, col = lane & 15, q = lane >> 4, ct = wave & 1, part = wave >> 1;
    const int h = blockIdx.y, p0 = (PARTS ? (int) blockIdx.x % cols : (int) blockIdx.x) * 32, pw = min(32, a.P - p0), N = a.N, inner = a.heads * a.P, ch = inner + 2 * a.groups * N, g = h / (a.heads / a.groups);
    const int n0 = part * NT * 16;                                 // first state row of this wave
    // this block's tokens [from, to).  The state in front of a part comes from a state that is fresh: one that a pass before left is where the last part's goes
    const int parts = !PARTS || e.pos0 > 0 ? 1 : (int) gridDim.x / cols, at = PARTS ? (int) blockIdx.x / cols : 0, chunks = (e.n + 15) / 16;
    if (at >= parts) return;
    auto border = [&](int k) { return k == 0 ? 0 : k >= parts ? e.n : min(chunks - 1, (int) ((float) chunks * (k == 1 ? cut.at[0] : k == 2 ? cut.at[1] : cut.at[2]) + 0.5f)) * 16; };
    const int from = border(at), to = border(at + 1);              // (inner borders lie in front of the last chunk: no part reaches behind the tokens, and the last is never empty)
    if (from >= to) return;
    float * st = a.state + (((size_t) e.seq * a.heads + h) * N) * a.P + p0;
    bamd_v4 S[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) { const int n = n0 + j * 16 + q * 4 + i, p = ct * 16 + col; S[j][i] = e.pos0 > 0 && n < N && p < pw ? st[(size_t) n * a.P + p] : 0.f; }
    const float D = a.D[h];
    // Chunks on their way, by the parity of the chunk.  Every load is unconditional (a row or column clamped into range, zeroed on its way to LDS): a branch around each costs more
    // than the chunk's arithmetic.  Thread: state row kn of the tokens kt, kt + KS, .., column xc of token xt, step size and decay of token col
    float bf[2][PF], cf[2][PF], xf[2], zf[2], fdt[2], fdec[2];
    const int kn = tid % NP, kt = tid / NP, xc = tid & 31, xt = tid >> 5;
    const uint32_t kb = (uint32_t) (inner + g * N + min(kn, N - 1)), kc = kb + (uint32_t) (a.groups * N), xo = (uint32_t) (h * a.P + p0 + min(xc, pw - 1));
    int end = to;                                                  // of the tokens that are gone through now
    auto request = [&](int t0, auto par, auto full) {
        constexpr int R = decltype(par)::value; constexpr bool F = decltype(full)::value;
        const int nt = end - t0;
        if (nt <= 0) return;
        const float * f = a.filtered + (size_t) (e.row0 + t0) * ch, * z = a.in + (size_t) (e.row0 + t0) * a.ld;
        if (nt >= 16) {
            const uint32_t r = (uint32_t) (kt * ch);
#pragma unroll
            for (int i = 0; i < PF; ++i) { const float * fi = f + (size_t) (i * KS) * ch; bf[R][i] = fi[r + kb]; if constexpr (F) cf[R][i] = fi[r + kc]; }
        } else {
#pragma unroll
            for (int i = 0; i < PF; ++i) { const uint32_t r = (uint32_t) (min(kt + i * KS, nt - 1) * ch); bf[R][i] = f[r + kb]; if constexpr (F) cf[R][i] = f[r + kc]; }
        }
        const int t = min(xt, nt - 1);
        xf[R] = f[(uint32_t) (t * ch) + xo];
        if constexpr (F) zf[R] = z[(uint32_t) (t * a.ld) + xo];
        const float * p = a.steps + ((size_t) (e.row0 + t0 + min(col, nt - 1)) * a.heads + h) * 2;
        fdt[R] = col < nt ? p[0] : 0.f; fdec[R] = col < nt ? p[1] : 1.f;
    };
    // data-parallel moves inside a row of sixteen lanes (row_shr, row_shl); a lane without a source gets 1
    auto moved = [](float v, auto ctrl) { return __int_as_float(__builtin_amdgcn_update_dpp(0x3f800000, __float_as_int(v), decltype(ctrl)::value, 0xf, 0xf, false)); };
    auto scan_up = [&](float v) {                                  // products of lanes 0 .. col
        v *= moved(v, std::integral_constant<int, 0x111>()); v *= moved(v, std::integral_constant<int, 0x112>());
        v *= moved(v, std::integral_constant<int, 0x114>()); return v * moved(v, std::integral_constant<int, 0x118>());
    };
    auto put = [&](int nt, auto par, auto full) {                  // nt: the chunk's tokens and those behind
        constexpr int w = decltype(par)::value; constexpr bool F = decltype(full)::value;
        if (nt >= 16 && N == NP) {
#pragma unroll
            for (int i = 0; i < PF; ++i) { Bs[w][(kt + i * KS) * LB + kn] = bf[w][i]; if constexpr (F) Cs[w][(kt + i * KS) * LB + kn] = cf[w][i]; }
        } else {
#pragma unroll
            for (int i = 0; i < PF; ++i) { const bool in = kn < N && kt + i * KS < nt; Bs[w][(kt + i * KS) * LB + kn] = in ? bf[w][i] : 0.f; if constexpr (F) Cs[w][(kt + i * KS) * LB + kn] = in ? cf[w][i] : 0.f; }
        }
        xf[w] = xc < pw && xt < nt ? xf[w] : 0.f;
        xs[w][xt * LX + xc] = xf[w];
        if (wave < 4) {                                            // row s = tid / 16: the products of the decays s + 1 .. t = col (zero above the diagonal)
            const int s = tid >> 4;
            const float v = scan_up(col > s ? fdec[w] : 1.f);
            dm[w][col * LD + s] = col < s ? 0.f : v;
        } else if (wave == 4) {                                    // up to each token, and behind it
            const float p = scan_up(fdec[w]);
            float f = fdec[w];
            f *= moved(f, std::integral_constant<int, 0x101>()); f *= moved(f, std::integral_constant<int, 0x102>());
            f *= moved(f, std::integral_constant<int, 0x104>()); f *= moved(f, std::integral_constant<int, 0x108>());
            f = moved(f, std::integral_constant<int, 0x101>());
            if (lane < 16) { dts[w][lane] = fdt[w]; pre[w][lane] = p; fd[w][lane] = f * fdt[w]; }
        }
    };
    // whole: outputs and state; the state alone is what a later part of the tokens starts from, in the same bits as long as neither takes a chunk again
    const std::integral_constant<bool, true> whole; const std::integral_constant<bool, false> state_only;
    auto state_chunk = [&](int t0, auto par) {
        constexpr int w = decltype(par)::value;
        const int nt = end - t0;
        request(t0 + 32, par, state_only);
        bamd_v4 T[NT];
        float ba[NT][4], xw[4], sum = 0.f;
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int i = 0; i < 4; ++i) ba[j][i] = Bs[w][(q * 4 + i) * LB + n0 + j * 16 + col];
        const bamd_v4 f4 = *(const bamd_v4 *) &fd[w][q * 4];
        const float all = pre[w][15];
#pragma unroll
        for (int i = 0; i < 4; ++i) xw[i] = xs[w][(q * 4 + i) * LX + ct * 16 + col] * f4[i];
        if (nt > 16) put(nt - 16, std::integral_constant<int, w ^ 1>(), state_only);
#pragma unroll
        for (int j = 0; j < NT; ++j) T[j] = S[j] * all;
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j) T[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(ba[j][i], xw[i], T[j], 0, 0, 0);
#pragma unroll
        for (int j = 0; j < NT; ++j) sum += (T[j][0] + T[j][1]) + (T[j][2] + T[j][3]);
        if (!__any(!(fabsf(sum) < INFINITY))) {
#pragma unroll
            for (int j = 0; j < NT; ++j) S[j] = T[j];
        } else for (int t = 0; t < 16; ++t) {
            const float d = t ? dm[w][t * LD + t - 1] : pre[w][0], xv = dts[w][t] * xs[w][t * LX + ct * 16 + col];
#pragma unroll
            for (int j = 0; j < NT; ++j) {
                const bamd_v4 B = *(const bamd_v4 *) &Bs[w][t * LB + n0 + j * 16 + q * 4];
#pragma unroll
                for (int i = 0; i < 4; ++i) S[j][i] = fmaf(d, S[j][i], B[i] * xv);
            }
        }
        __syncthreads();
    };
    auto chunk = [&](int t0, auto par) {
        constexpr int w = decltype(par)::value;
        const int nt = end - t0;
        const float xk = xf[w], zk = zf[w];
        request(t0 + 32, par, whole);
        bamd_v4 cr[NT], br[NT], gt = { 0, 0, 0, 0 }, g2 = { 0, 0, 0, 0 }, y = { 0, 0, 0, 0 }, y2 = { 0, 0, 0, 0 };
        bamd_v4 T[NT];                                                // the state behind the chunk
        float ba[NT][4], xw[4], xd[4];
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            cr[j] = *(const bamd_v4 *) &Cs[w][col * LB + n0 + j * 16 + q * 4]; br[j] = *(const bamd_v4 *) &Bs[w][col * LB + n0 + j * 16 + q * 4];
#pragma unroll
            for (int i = 0; i < 4; ++i) ba[j][i] = Bs[w][(q * 4 + i) * LB + n0 + j * 16 + col];
        }
        const bamd_v4 pr = *(const bamd_v4 *) &pre[w][q * 4], dv = *(const bamd_v4 *) &dm[w][col * LD + q * 4], d4 = *(const bamd_v4 *) &dts[w][q * 4], f4 = *(const bamd_v4 *) &fd[w][q * 4];
        const float all = pre[w][15];
#pragma unroll
        for (int i = 0; i < 4; ++i) { const float x = xs[w][(q * 4 + i) * LX + ct * 16 + col]; xd[i] = x * d4[i]; xw[i] = x * f4[i]; }
        if (nt > 16) put(nt - 16, std::integral_constant<int, w ^ 1>(), whole);       // (requested a chunk ago; its place was read before the last barrier)
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if (i & 1) { g2 = __builtin_amdgcn_mfma_f32_16x16x4f32(br[j][i], cr[j][i], g2, 0, 0, 0); y2 = __builtin_amdgcn_mfma_f32_16x16x4f32(cr[j][i], S[j][i], y2, 0, 0, 0); }
                else { gt = __builtin_amdgcn_mfma_f32_16x16x4f32(br[j][i], cr[j][i], gt, 0, 0, 0); y = __builtin_amdgcn_mfma_f32_16x16x4f32(cr[j][i], S[j][i], y, 0, 0, 0); }
            }
#pragma unroll
        for (int j = 0; j < NT; ++j) T[j] = S[j] * all;
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j) T[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(ba[j][i], xw[i], T[j], 0, 0, 0);
        y = (y + y2) * pr;
#pragma unroll
        for (int i = 0; i < 4; ++i) y = __builtin_amdgcn_mfma_f32_16x16x4f32((gt[i] + g2[i]) * dv[i], xd[i], y, 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 4; ++i) yp[w][part][(q * 4 + i) * LX + ct * 16 + col] = y[i];
        const float sum = (y[0] + y[1]) + (y[2] + y[3]);          // (looked at while the stores are under way; a sum that overflows by itself costs time, nothing else)
        if (!__any(!(fabsf(sum) < INFINITY))) {
#pragma unroll
            for (int j = 0; j < NT; ++j) S[j] = T[j];
        } else {
            for (int t = 0; t < min(nt, 16); ++t) {
                const float d = t ? dm[w][t * LD + t - 1] : pre[w][0], xv = dts[w][t] * xs[w][t * LX + ct * 16 + col];
                float y = 0.f;
#pragma unroll
                for (int j = 0; j < NT; ++j) {
                    const bamd_v4 B = *(const bamd_v4 *) &Bs[w][t * LB + n0 + j * 16 + q * 4], C = *(const bamd_v4 *) &Cs[w][t * LB + n0 + j * 16 + q * 4];
#pragma unroll
                    for (int i = 0; i < 4; ++i) { S[j][i] = fmaf(d, S[j][i], B[i] * xv); y = fmaf(C[i], S[j][i], y); }
                }
                y += __shfl_xor(y, 16); y += __shfl_xor(y, 32);
                if (q == 0) yp[w][part][t * LX + ct * 16 + col] = y;
            }
        }
        __syncthreads();
        const int o = xt * LX + xc;
        if (xt < nt && xc < pw) a.out[(size_t) (e.row0 + t0 + xt) * a.ldo + h * a.P + p0 + xc] = ((yp[w][0][o] + yp[w][1][o]) + (yp[w][2][o] + yp[w][3][o]) + D * xk) * silu_f(zk);
    };
    const std::integral_constant<int, 0> even; const std::integral_constant<int, 1> odd;
    if (PARTS && from > 0) {
        end = from;
        request(0, even, state_only); request(16, odd, state_only);
        put(end, even, state_only);
        __syncthreads();
        for (int t0 = 0; t0 < end; t0 += 32) { state_chunk(t0, even); if (t0 + 16 < end) state_chunk(t0 + 16, odd); }
        end = to;
    }
    request(from, even, whole); request(from + 16, odd, whole);
    put(end - from, even, whole);
    __syncthreads();
    for (int t0 = from; t0 < end; t0 += 32) { chunk(t0, even); if (t0 + 16 < end) chunk(t0 + 16, odd); }
    if (at + 1 < parts) return;
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) { const int n = n0 + j * 16 + q * 4 + i, p = ct * 16 + col; if (n < N && p < pw) st[(size_t) n * a.P + p] = S[j][i]; }
}
template <int PT, bool FOUR> static void step_go(const bamd_batch_dev & b, const bamd_ssm_args & a, hipStream_t s) {
    constexpr int GROUPS = 4 * 64 / (PT / 4);                      // 16 (64 columns), 32, 64
    const dim3 grid((a.P + PT - 1) / PT, a.heads, b.n_entries);
    const int npl = (a.N + GROUPS - 1) / GROUPS;
    if (npl <= 1) hipLaunchKernelGGL((ssm_step_kernel<PT, 1, FOUR>), grid, dim3(256), 0, s, b, a);
    else if (npl <= 2) hipLaunchKernelGGL((ssm_step_kernel<PT, 2, FOUR>), grid, dim3(256), 0, s, b, a);
    else if (npl <= 4) hipLaunchKernelGGL((ssm_step_kernel<PT, 4, FOUR>), grid, dim3(256), 0, s, b, a);
    else if constexpr (PT >= 32) {
        if (npl <= 8) hipLaunchKernelGGL((ssm_step_kernel<PT, 8, FOUR>), grid, dim3(256), 0, s, b, a);
        else if constexpr (PT >= 64) hipLaunchKernelGGL((ssm_step_kernel<PT, 16, FOUR>), grid, dim3(256), 0, s, b, a);
    }
}
static decltype(&ssm_chunk_kernel<1, false>) chunk_kernel(int N, int parts) {
    if (N <= 64) return parts > 1 ? ssm_chunk_kernel<1, true> : ssm_chunk_kernel<1, false>;
    if (N <= 128) return parts > 1 ? ssm_chunk_kernel<2, true> : ssm_chunk_kernel<2, false>;
    return parts > 1 ? ssm_chunk_kernel<4, true> : ssm_chunk_kernel<4, false>;
}
// max_n: most tokens any entry brings.  a.filtered [rows][channels] and a.steps [rows][heads][2] are scratch of prompts
int bamd_launch_ssm(const bamd_batch_dev & b, const bamd_ssm_args & a, int max_n, hipStream_t s) {
    if (a.N < 1 || a.N > 256 || a.taps < 1 || a.groups < 1 || a.heads % a.groups || max_n < 1) return 1;
    const int ch = a.heads * a.P + 2 * a.groups * a.N;
    if (max_n == 1) {
        // enough blocks for the chip; narrower blocks only as far as they are filled
        const long wide = (long) ((a.P + 63) / 64) * a.heads * b.n_entries;
        const int pt = a.P <= 16 || wide * 2 < 256 ? 16 : a.P <= 32 || wide < 256 ? 32 : 64;
        if (a.taps == 4) { if (pt == 16) step_go<16, true>(b, a, s); else if (pt == 32) step_go<32, true>(b, a, s); else step_go<64, true>(b, a, s); }
        else { if (pt == 16) step_go<16, false>(b, a, s); else if (pt == 32) step_go<32, false>(b, a, s); else step_go<64, false>(b, a, s); }
        return 0;
    }
    if (!a.filtered || !a.steps) return 1;
    const int cols = (a.P + 31) / 32, blocks = cols * a.heads * b.n_entries;
    const int parts = max_n < 64 ? 1 : std::max(1, std::min(4, 256 / blocks));      // (of fewer tokens they are level)
    ssm_cut cut = { { 1.f, 1.f, 1.f } };
    for (int k = 1; k < parts; ++k) cut.at[k - 1] = (1.f - powf(SSM_AGAIN, (float) k)) / (1.f - powf(SSM_AGAIN, (float) parts));
    const dim3 cg((ch + 255) / 256, (b.rows + SSM_STRIP - 1) / SSM_STRIP), grid(cols * parts, a.heads, b.n_entries);
    if (a.taps == 4) hipLaunchKernelGGL(ssm_conv_kernel<true>, cg, dim3(256), 0, s, b, a); else hipLaunchKernelGGL(ssm_conv_kernel<false>, cg, dim3(256), 0, s, b, a);
    hipLaunchKernelGGL(chunk_kernel(a.N, parts), grid, dim3(512), 0, s, b, a, cols, cut);
    return 0;
}
int bamd_ssm_chunk_blocks(int N, int parts) {
    int n = 0;
    return hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, (const void *) chunk_kernel(N, parts), 512, 0) == hipSuccess ? n : -1;
}
