// bamd_pair.hip — decoded tokens through two mixers side by side, attention over cached keys and values (bamd_kv_device.h) and gated linear attention (bamd_gla_device.h): each is
// a chain of dependent reads that leaves most of the chip idle, so that their blocks share a launch — where keys are few everything of a token, otherwise the shares of the keys and the state updates first, then the sums over
// the shares and the norms of the heads.
#include "bamd_kv_device.h"
#include "bamd_gla_device.h"
#include <algorithm>
#include <string.h>

// block (attention shares x groups, then value columns, PT at a time, x heads; row)
template <typename T, int ND, int PT, int NPL>
__global__ void __launch_bounds__(256, ND <= 4 ? 2 : 1) kv_gla_step_kernel(bamd_batch_dev b, bamd_kv_args kv, bamd_gla_args gla, float * part_o, float * part_ml, int splits, int attn) {
    extern __shared__ __align__(16) unsigned char lds[];
    const int x = blockIdx.x, row = blockIdx.y;
    if (x < attn) { kv_decode_block<T, ND>(b, kv, x / (attn / splits), splits, x % (attn / splits), row, part_o, part_ml, lds); return; }
    const int cols = (gla.Pp + PT - 1) / PT, i = x - attn, h = i / cols;
    const bamd_entry e = b.ent[row];
    float * st = gla.state + ((size_t) e.seq * gla.heads + h) * gla.Np * gla.Pp;
    gla_scan_block<PT, NPL, GLA_STEP>(gla, h, (i % cols) * PT, row, 1, e.pos0 > 0 ? st : nullptr, st, nullptr, lds);
}
// block (head of the attention, then sixteen heads of the recurrence; row)
template <typename T> __global__ void __launch_bounds__(256) kv_gla_finish_kernel(bamd_kv_args kv, bamd_gla_args gla, const float * part_o, const float * part_ml, int splits) {
    if ((int) blockIdx.x < kv.heads) kv_combine_block<T>(kv, blockIdx.x, blockIdx.y, part_o, part_ml, splits);
    else gla_norm_block<T>(gla, (blockIdx.x - kv.heads) * 16, blockIdx.y);
}

template <typename T, int ND, int PT, int NPL>
static int pair_go(const bamd_batch_dev & b, const bamd_kv_args & kv, const bamd_gla_args & gla, float * po, float * pm, int splits, hipStream_t s) {
    constexpr size_t lk = KvDecodeLds<T, ND>::bytes, lg = GlaShape<PT, NPL, GLA_STEP>::lds, lds = lk > lg ? lk : lg;
    const int attn = splits * bamd_kv_groups(kv), cols = (gla.Pp + PT - 1) / PT;
    hipLaunchKernelGGL((kv_gla_step_kernel<T, ND, PT, NPL>), dim3(attn + gla.heads * cols, b.rows), dim3(256), lds, s, b, kv, gla, po, pm, splits, attn);
    hipLaunchKernelGGL(kv_gla_finish_kernel<T>, dim3(kv.heads + (gla.heads + 15) / 16, b.rows), dim3(256), 0, s, kv, gla, po, pm, splits);
    return 0;
}
// state rows per lane: PT / 16 for every 64 key channels
template <typename T, int ND, int PT>
static int pair_npl(const bamd_batch_dev & b, const bamd_kv_args & kv, const bamd_gla_args & gla, float * po, float * pm, int splits, hipStream_t s) {
    if (gla.Np <= 64) return pair_go<T, ND, PT, PT / 16>(b, kv, gla, po, pm, splits, s);
    if (gla.Np <= 128) return pair_go<T, ND, PT, PT / 8>(b, kv, gla, po, pm, splits, s);
    return pair_go<T, ND, PT, PT / 4>(b, kv, gla, po, pm, splits, s);
}
template <typename T, int ND>
static int pair_pt(const bamd_batch_dev & b, const bamd_kv_args & kv, const bamd_gla_args & gla, float * po, float * pm, int splits, hipStream_t s) {
    switch (bamd_gla_step_columns(gla, b.rows)) {
        case 16: return pair_npl<T, ND, 16>(b, kv, gla, po, pm, splits, s);
        case 32: return pair_npl<T, ND, 32>(b, kv, gla, po, pm, splits, s);
    }
    return pair_npl<T, ND, 64>(b, kv, gla, po, pm, splits, s);
}
template <typename T>
static int pair_nd(const bamd_batch_dev & b, const bamd_kv_args & kv, const bamd_gla_args & gla, float * po, float * pm, int splits, hipStream_t s) {
    switch (kv.D) {
        case 32: return pair_pt<T, 1>(b, kv, gla, po, pm, splits, s);
        case 64: return pair_pt<T, 2>(b, kv, gla, po, pm, splits, s);
        case 128: return pair_pt<T, 4>(b, kv, gla, po, pm, splits, s);
        case 256: return pair_pt<T, 8>(b, kv, gla, po, pm, splits, s);
    }
    return 1;
}
int bamd_launch_kv_gla_decode(int act, const bamd_batch_dev & b, const bamd_kv_args & kv, const bamd_gla_args & gla, float * po, float * pm, int splits, hipStream_t s) {
    if (splits < 1 || splits > 64 || b.rows != b.n_entries || !bamd_kv_valid(kv) || !bamd_gla_valid(gla)) return 1;
    return act == BAMD_ACT_F32 ? pair_nd<float>(b, kv, gla, po, pm, splits, s) : pair_nd<bamd_bf>(b, kv, gla, po, pm, splits, s);
}

// Both mixers of a decoded token in one launch: a block per group of heads that share keys walks all of them (seven waves, half pages in turn, and one for the token's own) and writes its heads' results, a block per head of the
// recurrence takes all its columns, norm and gate.  The two launches above become one where the keys are few.  Two half pages of a wave on their way at once, or twelve waves, spill (5 % of a step slower).
// block (group of the attention, then head of the recurrence; row); without one of them (attn or heads 0) the other alone
template <typename T, int ND, int PT, int NPL>
__global__ void __launch_bounds__(512) kv_gla_one_kernel(bamd_batch_dev b, bamd_kv_args kv, bamd_gla_args gla, int attn) {
    extern __shared__ __align__(16) unsigned char lds[];
    const int x = blockIdx.x, row = blockIdx.y;
    if (x < attn) { kv_decode_block<T, ND, 8, true>(b, kv, 0, 1, x, row, nullptr, nullptr, lds); return; }
    const int h = x - attn;
    const bamd_entry e = b.ent[row];
    gla_head_block<T, PT, NPL>(gla, h, row, e.pos0 == 0, gla.state + ((size_t) e.seq * gla.heads + h) * gla.Np * gla.Pp, lds);
}
template <typename T, int ND, int PT, int NPL>
static void one_go(const bamd_batch_dev & b, const bamd_kv_args & kv, const bamd_gla_args & gla, int attn, hipStream_t s) {
    constexpr size_t lk = KvDecodeLds<T, ND, 8>::bytes, lg = GlaHead<T, PT, NPL>::lds, lds = lk > lg ? lk : lg;
    hipLaunchKernelGGL((kv_gla_one_kernel<T, ND, PT, NPL>), dim3(attn + gla.heads, b.rows), dim3(512), lds, s, b, kv, gla, attn);
}
template <typename T, int ND>
static void one_pick(const bamd_batch_dev & b, const bamd_kv_args & kv, const bamd_gla_args & gla, int attn, hipStream_t s) {
    if (gla.Pp <= 64) { if (gla.Np <= 64) one_go<T, ND, 64, 2>(b, kv, gla, attn, s); else one_go<T, ND, 64, 4>(b, kv, gla, attn, s); }
    else if (gla.Np <= 64) one_go<T, ND, 128, 4>(b, kv, gla, attn, s);
    else one_go<T, ND, 128, 8>(b, kv, gla, attn, s);
}
template <typename T> static int one_nd(const bamd_batch_dev & b, const bamd_kv_args & kv, const bamd_gla_args & gla, int attn, hipStream_t s) {
    if (kv.D == 32) one_pick<T, 1>(b, kv, gla, attn, s); else if (kv.D == 64) one_pick<T, 2>(b, kv, gla, attn, s); else one_pick<T, 4>(b, kv, gla, attn, s);
    return 0;
}
bool bamd_kv_gla_one_valid(const bamd_kv_args * kv, const bamd_gla_args * gla) { return (!kv || (bamd_kv_valid(*kv) && (kv->D == 32 || kv->D == 64 || kv->D == 128))) && (!gla || (bamd_gla_valid(*gla) && gla->Np <= 128 && gla->Pp <= 128)); }
// A block's seven waves take 224 keys at a time, and one time is what the second launch costs (5.8 us a layer with its gap); eight bfloat16 rows can afford two (six are level).  Steps of eight layers, us, two launches and
// one: width 1024, one row behind 20 positions 296 | 264, 205 309 | 291; twelve rows behind 150 404 | 372; 2048, one row 205 416 | 397, 240 416 | 417, 600 420 | 478; six rows 240 515 | 496, 400 514 | 515;
// sixteen rows 400 616 | 605; 4096, one row 45 857 | 817, 205 867 | 841; eight rows 400 1071 | 1038; 62 rows 25 1956 | 1918.  32-bit: 2048, one row 110 488 | 462, 205 490 | 479, 235 489 | 508; 40 rows 40
// 1431 | 1357; 4096, six rows 205 1333 | 1293
bool bamd_kv_gla_one_launch(int act, const bamd_kv_args & kv, const bamd_gla_args & gla, int rows, int most) {
    const bool f32 = act == BAMD_ACT_F32;
    return most > 0 && rows <= (f32 ? 48 : 64) && bamd_kv_gla_one_valid(&kv, &gla) && std::min<long>(most, (long) kv.window + kv.keep) <= (!f32 && rows >= 8 ? 448 : 224);
}
int bamd_launch_kv_gla_one(int act, const bamd_batch_dev & b, const bamd_kv_args * kv, const bamd_gla_args * gla, hipStream_t s) {
    bamd_kv_args k; bamd_gla_args g;
    memset((void *) &k, 0, sizeof k); memset((void *) &g, 0, sizeof g);
    k.D = 32;
    if (b.rows != b.n_entries || (!kv && !gla) || !bamd_kv_gla_one_valid(kv, gla)) return 1;
    if (kv) k = *kv;
    if (gla) g = *gla;
    const int attn = kv ? bamd_kv_groups(*kv) : 0;
    return act == BAMD_ACT_F32 ? one_nd<float>(b, k, g, attn, s) : one_nd<bamd_bf>(b, k, g, attn, s);
}
