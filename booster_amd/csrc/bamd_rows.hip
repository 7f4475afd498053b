// bamd_rows.hip — row-wise mechanisms of the configured layer stacks, one block per row: embedding with learned positions, residual sum with the norm of the
// sublayer's output and token shift (or layer norms in front and behind), PolyNorm, clamped gated unit, grouped norm, the model's last norm, arg-max, and the device side of the greedy loop.  With a single row the same
// device functions run as the prologue of the product behind them (bamd_dense.hip).
#include "bamd_dense_device.h"
#include <algorithm>

// columns i0 .. i0 + 3
__device__ __forceinline__ void embed_piece(int i0, int row, int t, int p, const uint16_t * __restrict__ embd, const uint16_t * __restrict__ pos, float scale, int E, int V, float * __restrict__ x) {
    t = t < 0 ? 0 : t >= V ? V - 1 : t;
    const uint16_t * er = embd + (size_t) t * E, * pr = pos ? pos + (size_t) p * E : nullptr;
    if (i0 + 3 < E && (E & 3) == 0) {
        const uint2 u = *(const uint2 *) (er + i0), w = pr ? *(const uint2 *) (pr + i0) : uint2{ 0, 0 };
        *(bamd_v4 *) (x + (size_t) row * E + i0) = bamd_v4{ bf_lo(u.x) * scale + bf_lo(w.x), bf_hi(u.x) * scale + bf_hi(w.x), bf_lo(u.y) * scale + bf_lo(w.y), bf_hi(u.y) * scale + bf_hi(w.y) };
    } else for (int i = i0; i < min(i0 + 4, E); ++i) x[(size_t) row * E + i] = bf_f(er[i]) * scale + (pr ? bf_f(pr[i]) : 0.f);
}
__global__ void __launch_bounds__(256) embed_rows_kernel(bamd_batch_dev b, const uint16_t * __restrict__ embd, const uint16_t * __restrict__ pos, float scale, int E, int V, float * __restrict__ x) {
    const int row = blockIdx.y;
    const bamd_entry e = b.ent[b.row_entry[row]];
    embed_piece(blockIdx.x * 1024 + threadIdx.x * 4, row, b.tokens[row], e.pos0 + (row - e.row0), embd, pos, scale, E, V, x);
}
__device__ __forceinline__ int32_t box_ld(const int32_t * p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM); }
// The step's descriptors and tokens come out of host memory here: a copy engine in front of the step, and one behind it, were 40 us of a token's 465 (width 2048).  A block per row, one lane of
// which reads its token and position (two independent reads over the bus), the first block the descriptors of all rows.  Every wave of a block per 1024 columns reading them by itself, they were
// 512 reads for sixteen rows of 4096: 27 us, now 7; one row of 2048 9.6, now 6.5
__global__ void __launch_bounds__(1024) step_open_kernel(const bamd_step_box * box, bamd_step_dev d, const uint16_t * __restrict__ embd, const uint16_t * __restrict__ pos, float scale, int E, int V, float * __restrict__ x) {
    __shared__ int32_t at[2];
    const int row = blockIdx.x, tid = threadIdx.x;
    if (tid == 0) { const int32_t t = box_ld(&box->in.tok[row]), p = pos ? box_ld(&box->in.ent[row].pos0) : 0; at[0] = t; at[1] = p; }
    if (row == 0) {
        const int n = gridDim.x, words = n * (int) (sizeof(bamd_entry) / 4), by = blockDim.x;
        for (int i = tid; i < words; i += by) ((int32_t *) d.ent)[i] = box_ld((const int32_t *) box->in.ent + i);
        for (int i = tid; i < n; i += by) { d.tokens[i] = box_ld(&box->in.tok[i]); d.row_entry[i] = i; d.want[i] = i; }
        if (tid == by - 1) d.count_serial[1] = (uint32_t) box_ld((const int32_t *) &box->in.serial);
    }
    __syncthreads();
    for (int i0 = tid * 4; i0 < E; i0 += blockDim.x * 4) embed_piece(i0, row, at[0], at[1], embd, pos, scale, E, V, x);
}
// n floats to host memory; the block that ends last tells the host.  Every thread's stores are out before its block counts
__global__ void __launch_bounds__(256) step_close_kernel(const float * __restrict__ logits, size_t n, float * __restrict__ host, uint32_t * done, uint32_t * count_serial) {
    const size_t stride = (size_t) gridDim.x * 256, i0 = (size_t) blockIdx.x * 256 + threadIdx.x;
    for (size_t i = i0; i < n / 4; i += stride) *(bamd_v4 *) (host + i * 4) = *(const bamd_v4 *) (logits + i * 4);
    for (size_t i = n / 4 * 4 + i0; i < n; i += stride) host[i] = logits[i];
    __threadfence_system();
    __syncthreads();
    if (threadIdx.x) return;
    if (__hip_atomic_fetch_add(count_serial, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) + 1 < gridDim.x) return;
    count_serial[0] = 0;
    __threadfence_system();
    __hip_atomic_store(done, count_serial[1], __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}
template <typename T, bool ONE> __global__ void __launch_bounds__(1024) residual_rows_kernel(bamd_batch_dev b, bamd_residual_args a) {
    __shared__ float red[64];
    residual_row<T, false, ONE>(b, a, blockIdx.x, row_out<T>(a.h, blockIdx.x, a.ldh, a.cb), true, red);
}
template <typename T, bool ONE> __global__ void __launch_bounds__(1024) final_rows_kernel(bamd_residual_args a, const int32_t * want, const float * gf) {
    __shared__ float red[64];
    final_row<T, ONE>(a, want[blockIdx.x], gf, row_out<T>(a.h, blockIdx.x, a.ldh, a.cb), red);
}
template <typename T, bool ONE> __global__ void __launch_bounds__(1024) layer_rows_kernel(bamd_residual_args a, const int32_t * want, const float * gi) {
    __shared__ float red[64];
    const int row = want ? want[blockIdx.x] : blockIdx.x;
    layer_row<T, ONE>(a, row, gi, row_out<T>(a.h, blockIdx.x, a.ldh, a.cb), !want, red);
}
// block (1024 columns, row)
template <typename T> __global__ void __launch_bounds__(256) glu_rows_kernel(bamd_glu_args a) { glu_row<T>(a, blockIdx.y, row_out<T>(a.h, blockIdx.y, a.ldh, a.cb), blockIdx.x * 1024, min(a.ldh, (int) blockIdx.x * 1024 + 1024)); }
template <typename T, bool ONE> __global__ void __launch_bounds__(1024) poly_rows_kernel(bamd_poly_args a) {
    __shared__ float red[64];
    poly_row<T, ONE>(a, blockIdx.x, row_out<T>(a.h, blockIdx.x, a.ldh, a.cb), red);
}
template <typename T> __global__ void __launch_bounds__(1024) group_norm_rows_kernel(bamd_group_norm_args a) {
    __shared__ float inv[BAMD_MAX_NORM_GROUPS + 16];
    group_norm_row<T>(a, blockIdx.x, row_out<T>(a.h, blockIdx.x, a.ldh, a.cb), inv);
}
// block (part, row); keys must be zero
__global__ void __launch_bounds__(256) argmax_rows_kernel(const float * __restrict__ logits, int V, unsigned long long * keys) {
    __shared__ unsigned long long wk[4];
    const float * l = logits + (size_t) blockIdx.y * V;
    unsigned long long best = 0ull;
    for (int i = blockIdx.x * 256 + threadIdx.x; i < V; i += gridDim.x * 256) {
        const float f = l[i];
        if (f != f) continue;
        const unsigned int u = __float_as_uint(f), o = (u & 0x80000000u) ? ~u : (u | 0x80000000u);
        const unsigned long long k = ((unsigned long long) o << 32) | (0xffffffffu - (unsigned int) i);
        best = k > best ? k : best;
    }
    for (int o = 32; o > 0; o >>= 1) { const unsigned long long k = __shfl_xor(best, o); best = k > best ? k : best; }
    if ((threadIdx.x & 63) == 0) wk[threadIdx.x >> 6] = best;
    __syncthreads();
    if (threadIdx.x == 0) { for (int w = 1; w < 4; ++w) best = wk[w] > best ? wk[w] : best; if (best) atomicMax(keys + blockIdx.y, best); }
}
__global__ void __launch_bounds__(64) clear_keys_kernel(unsigned long long * keys, int n) { for (int i = threadIdx.x; i < n; i += 64) keys[i] = 0ull; }
__global__ void __launch_bounds__(64) advance_kernel(bamd_entry * ent, int32_t * tokens, unsigned long long * keys, int n, int32_t * out, int ldo, int32_t * step, int advance, int V) {
    const int i = threadIdx.x, at = step ? *step : 0;
    for (int j = i; j < n; j += 64) {
        const uint32_t id = 0xffffffffu - (uint32_t) (keys[j] & 0xffffffffull);
        const int t = id < (uint32_t) V ? (int) id : 0;
        if (out && at < ldo) out[(size_t) j * ldo + at] = t;
        if (tokens) tokens[j] = t;
        if (advance) keys[j] = 0ull;                              // for the arg-max at this step's end
        if (advance) { if (at > 0) { ent[j].pos0 += 1; ent[j].par ^= 1; } }
    }
    __syncthreads();
    if (i == 0 && step) *step = at + 1;
}

static dim3 row_block(int n) { return dim3(n > 1024 ? 1024 : 256); }
// Rows that two pieces of four floats per thread hold (RowRegs<2>): no more waves than that takes, since every sum over the row waits for all of them
// (layer norms of six rows of 2048: 6.6 -> 5.5 us, of 2048 rows of 4096: 32 -> 23 us; up to 1024 threads before; six rows of 2052: 5.3 -> 4.8 us, 14.1 on the 256 threads that fall four floats short).  Other lengths are held one float
// at a time, on 1024 threads while that many blocks are resident at once (six rows of 4098: 6.4 us, 6.8 on 576 threads; of 2050 6.2, 5.7 on 320; read again for every sum they took 9.8 and 7.4)
int bamd_norm_threads(int n, int rows) { return (n & 3) && rows <= 512 ? (int) row_block(n).x : std::min(1024, std::max(256, ((n + 7) / 8 + 63) / 64 * 64)); }
static dim3 sum_block(int n, int rows) { return dim3(bamd_norm_threads(n, rows)); }
void bamd_launch_embed_rows(const bamd_batch_dev & b, const uint16_t * embd, const uint16_t * pos, float scale, int E, int V, float * x, hipStream_t s) {
    hipLaunchKernelGGL(embed_rows_kernel, dim3((E + 1023) / 1024, b.rows), dim3(256), 0, s, b, embd, pos, scale, E, V, x);
}
void bamd_launch_step_open(const bamd_step_box * box, int rows, const bamd_step_dev & d, const uint16_t * embd, const uint16_t * pos, float scale, int E, int V, float * x, hipStream_t s) {
    hipLaunchKernelGGL(step_open_kernel, dim3(rows), dim3(std::min(1024, std::max(128, ((E + 3) / 4 + 63) / 64 * 64))), 0, s, box, d, embd, pos, scale, E, V, x);
}
// a block per 4096 floats, up to 128: a row of 32 000 goes out at the bus's rate
void bamd_launch_step_close(const float * logits, size_t n, float * host, bamd_step_box * box, uint32_t * count_serial, hipStream_t s) {
    const size_t blocks = (n + 4095) / 4096;
    hipLaunchKernelGGL(step_close_kernel, dim3((unsigned) (blocks < 1 ? 1 : blocks > 128 ? 128 : blocks)), dim3(256), 0, s, logits, n, host, &box->done, count_serial);
}
// by the compile-time kinds: operands, and whether a row's length is a multiple of four
#define ROWS_GO(KERNEL_, N_, ROWS_, BLOCK_, ...) do { \
        if (act == BAMD_ACT_F32) { if ((N_) & 3) hipLaunchKernelGGL((KERNEL_<bamd_s3, true>), dim3(ROWS_), BLOCK_, 0, s, __VA_ARGS__); else hipLaunchKernelGGL((KERNEL_<bamd_s3, false>), dim3(ROWS_), BLOCK_, 0, s, __VA_ARGS__); } \
        else if ((N_) & 3) hipLaunchKernelGGL((KERNEL_<bamd_bf, true>), dim3(ROWS_), BLOCK_, 0, s, __VA_ARGS__); else hipLaunchKernelGGL((KERNEL_<bamd_bf, false>), dim3(ROWS_), BLOCK_, 0, s, __VA_ARGS__); } while (0)
void bamd_launch_residual_rows(int act, const bamd_batch_dev & b, const bamd_residual_args & a, hipStream_t s) {
    if (a.norm == BAMD_NORM_LAYER) ROWS_GO(layer_rows_kernel, a.E, b.rows, sum_block(a.E, b.rows), a, nullptr, a.gi);
    else ROWS_GO(residual_rows_kernel, a.E, b.rows, sum_block(a.E, b.rows), b, a);
}
void bamd_launch_final_rows(int act, const bamd_residual_args & a, const int32_t * want, int n_want, const float * gf, hipStream_t s) {
    if (a.norm == BAMD_NORM_LAYER) ROWS_GO(layer_rows_kernel, a.E, n_want, sum_block(a.E, n_want), a, want, gf);
    else ROWS_GO(final_rows_kernel, a.E, n_want, sum_block(a.E, n_want), a, want, gf);
}
void bamd_launch_poly_rows(int act, int rows, const bamd_poly_args & a, hipStream_t s) {
    ROWS_GO(poly_rows_kernel, a.F, rows, row_block(a.F), a);
}
void bamd_launch_glu_rows(int act, int rows, const bamd_glu_args & a, hipStream_t s) {
    if (act == BAMD_ACT_F32) hipLaunchKernelGGL(glu_rows_kernel<bamd_s3>, dim3((a.ldh + 1023) / 1024, rows), dim3(256), 0, s, a);
    else hipLaunchKernelGGL(glu_rows_kernel<bamd_bf>, dim3((a.ldh + 1023) / 1024, rows), dim3(256), 0, s, a);
}
void bamd_launch_group_norm_rows(int act, int rows, const bamd_group_norm_args & a, hipStream_t s) {
    if (act == BAMD_ACT_F32) hipLaunchKernelGGL(group_norm_rows_kernel<bamd_s3>, dim3(rows), row_block(a.n), 0, s, a);
    else hipLaunchKernelGGL(group_norm_rows_kernel<bamd_bf>, dim3(rows), row_block(a.n), 0, s, a);
}
void bamd_launch_argmax_rows(const float * logits, int n, int V, unsigned long long * keys, bool clear, hipStream_t s) {
    if (clear) hipLaunchKernelGGL(clear_keys_kernel, dim3(1), dim3(64), 0, s, keys, n);
    hipLaunchKernelGGL(argmax_rows_kernel, dim3(V > 8192 ? 32 : 4, n), dim3(256), 0, s, logits, V, keys);
}
void bamd_launch_advance(bamd_entry * ent, int32_t * tokens, unsigned long long * keys, int n, int32_t * out, int ldo, int32_t * step, int advance, int V, hipStream_t s) {
    hipLaunchKernelGGL(advance_kernel, dim3(1), dim3(64), 0, s, ent, tokens, keys, n, out, ldo, step, advance, V);
}
