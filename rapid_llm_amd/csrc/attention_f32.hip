// Paged causal attention in true float32 on the matrix cores' float32 instruction
// (v_mfma_f32_16x16x4_f32), compiled for one head size RL_HEAD_DIM (a multiple of 16).
//
// One workgroup of four waves per (tile of 16 rows, kv head).  Rows are (token, query head of
// the kv group) pairs of ONE request, so grouped heads and neighbouring tokens share every key
// that is read.  The key tiles are dealt to the waves by their absolute index (tile i goes to
// wave i % 4), each wave keeps a softmax state of its own, and the four states are folded in
// the order of the waves: a single token's long context is then read by four waves at once.  As in the bfloat16 kernels the transposed products are computed,
//   S^T[keys, rows] = K[keys, d] Q^T[d, rows],   O^T[d, rows] += V^T[d, keys] P^T[keys, rows],
// which leaves a lane with the scores of keys 4g .. 4g + 3 of its own row: exactly its
// operand of the second product, whose other operand is one 16-byte read of the transposed
// value cache.  Softmax state is one scalar per lane.
//
// A row's result does not depend on the tile it falls in, on the other rows there, or on how
// a prompt was cut into steps: keys are taken in tiles of 16 at absolute positions 0, 16, ..,
// in spans of SPAN keys at absolute positions.  Within a span each wave takes its tiles in ascending
// order, beginning with an empty state; a wave's states of the spans are folded in their order, and then
// the waves'.  Within a tile the order of every sum is fixed by the key's position; a tile that holds
// no visible key of a row leaves that row's state as it is, exactly (factor 1, terms 0), and so does
// a span or a wave without visible keys in the fold.  A launch of few tiles (decoding) may therefore
// give every span to a workgroup of its own, which leaves its waves' states to a second kernel that
// folds them in the same order: the same bits.
//
// What bounds it: whole contexts of 2,048 keys, 32 query and 8 kv heads of 128 channels, take 404 us (85 TFLOP/s;
// 5,000 keys 91) called alone, and 471 a layer in the prompt step under the profiler, where nothing of them is near.  The float32 matrix instructions hold the vector units for 53% of that, their rate, and the
// other vector instructions for 36%, the weights of a tile above all; they do not overlap.  Two tiles of rows a
// workgroup, which halve the keys that are read, leave one wave a SIMD and took 428 us.  Before, a tile's entry of the
// block table was asked for and waited for with its keys and with its values, both behind every load in flight, at a
// position that took a division, and the maximum and the sum of a row went through LDS: 514 us, 591 in the step.  Masked keys contribute exactly zero
// (rapid_llm/kernels/ops/attention/flashdecoding.py:223-237); scores are (q . k) / sqrt(d)
// (rapid_llm/modules/attention.py:62), softmax over keys in float32
// (rapid_llm/kernels/ops/attention/flashattention2_nopad.py:138-168).
#include "common.h"

#ifndef RL_HEAD_DIM
#error "compile with -DRL_HEAD_DIM=<head size>"
#endif

namespace f32attn {

constexpr int D = RL_HEAD_DIM;
constexpr int DB = D / 16;  // 16-channel chunks of the first product = blocks of the output
constexpr int AW = 4;       // waves per workgroup: key tile i belongs to wave i % AW
// Keys a span.  Eight requests of 512 to 1,536 keys of the 8B shape: 64 workgroups that walked whole
// contexts took 65 us a layer, the latency of their chain of tiles, the step 8.95 ms; spans in workgroups
// of their own leave it at 7.80 ms.  Spans of 256 keys rather than 512 take a single request of 1,000 keys
// of the 0.6B shape from 2.19 to 1.97 ms a step and cost a prompt of 2,048 tokens 0.3%, for a fold every
// four tiles of a wave; of 128 they cost it 4%.
constexpr int SPAN = 256;
constexpr int STATE = D + 2;  // floats a (row, wave, span) state takes in memory: sums, maximum, sum of weights
// floats that the states of a wave's rows take, whole lines of 128 bytes
__host__ __device__ constexpr int wave_states(int held) { return (held * STATE + 31) / 32 * 32; }
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ inline f32x4 ld4(const float* p) { return *reinterpret_cast<const f32x4*>(p); }

// the four lanes (r, g = 0..3) that share a row: the same bits in each of them
// (exchanged between registers: through LDS, as a shuffle goes, each step waits for a round trip)
__device__ inline float row_max(float v) {
    const unsigned u = __float_as_uint(v);
    const auto a = __builtin_amdgcn_permlane16_swap(u, u, false, false);
    const unsigned w = __float_as_uint(fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1])));
    const auto b = __builtin_amdgcn_permlane32_swap(w, w, false, false);
    return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
__device__ inline float row_sum(float v) {
    const unsigned u = __float_as_uint(v);
    const auto a = __builtin_amdgcn_permlane16_swap(u, u, false, false);
    const unsigned w = __float_as_uint(__uint_as_float(a[0]) + __uint_as_float(a[1]));
    const auto b = __builtin_amdgcn_permlane32_swap(w, w, false, false);
    return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

// A position of the cache that walks on by the keys between two tiles of a wave, without a division.
struct Walk {
    int key, page, off;
    __device__ inline void step(int keys, int pages, int offs, int page_size) {
        key += keys;
        page += pages;
        off += offs;
        if (off >= page_size) {
            off -= page_size;
            ++page;
        }
    }
};

// (m, l, acc) folded with the state of later keys, (m2, l2, acc2); written out so that every kernel
// rounds alike.  `none`: neither has seen a key.
struct Fold {
    float m, fa, fb;
    bool none;
};
__device__ inline Fold fold_of(float m, float m2) {
    Fold f;
    f.m = fmaxf(m, m2);
    f.none = f.m == -INFINITY;
    f.fa = f.none ? 1.f : expf(m - f.m);
    f.fb = f.none ? 0.f : expf(m2 - f.m);
    return f;
}
__device__ inline float fold_sum(float x, float x2, const Fold& f) { return fmaf(x2, f.fb, x * f.fa); }

// tile_info: [tiles][3] = index of the request's first token in the step, its tokens in the
// step, first row of the tile.  The request's first position is read from `positions`.
// SPLIT: blockIdx.z takes `per` spans; states[tile][kv head][span][wave] of wave_states take the place of `out`, with
// as many rows as a tile of the launch has at most (`held`: a decoding request's tile has its query heads).
template <bool SPLIT>
__global__ __launch_bounds__(AW* RL_WAVE) void attn_f32_kernel(
    const float* __restrict__ q, const float* __restrict__ k_cache,
    const float* __restrict__ v_cache, float* __restrict__ out, float* __restrict__ states,
    const int* __restrict__ tile_info, const int* __restrict__ positions,
    const int* __restrict__ token_slot, const int* __restrict__ block_table, int table_stride,
    int page_size, int nq, int nkv, int window, float scale, int spans, int per, int held) {
    // Whole contexts: neighbouring workgroups have different kv heads, so that with eight of them each of the
    // chip's dies keeps one in its L2, and the last tiles, which have the most keys, begin first.
    const int tile = SPLIT ? blockIdx.x : gridDim.x / nkv - 1 - blockIdx.x / nkv;
    const int hk = SPLIT ? blockIdx.y : blockIdx.x % nkv;
    const int G = nq / nkv;
    const int at = tile_info[3 * tile], n = tile_info[3 * tile + 1], row0 = tile_info[3 * tile + 2];
    __shared__ float fold_ml[AW - 1][2][RL_WAVE];
    __shared__ f32x4 fold_acc[AW - 1][DB][RL_WAVE];
    const int lane = threadIdx.x & (RL_WAVE - 1);
    const int wave = threadIdx.x / RL_WAVE;
    const int r16 = lane & 15;
    const int g = lane >> 4;
    const int start = positions[at];
    const int* table = block_table + (size_t)token_slot[at] * table_stride;

    const int rows = n * G;
    const int row = row0 + r16;
    const bool row_ok = row < rows;
    const int tok = (row_ok ? row : rows - 1) / G;
    const int head = hk * G + (row_ok ? row : rows - 1) % G;
    const int pos = start + tok;
    const int kend = pos + 1;
    const int kstart = (window > 0 && pos - window + 1 > 0) ? pos - window + 1 : 0;

    // the keys any row of the tile sees: from the first row's first key (rows ascend with
    // the tokens), in whole tiles of 16, up to the last row's own position
    const int first_pos = start + row0 / G;
    const int last_pos = start + (min(rows, row0 + 16) - 1) / G;
    const int first_key = (window > 0 && first_pos - window + 1 > 0) ? first_pos - window + 1 : 0;
    const int lo = first_key & ~15;
    const int hi = last_pos + 1;  // keys below hi are in the cache
    // the keys this workgroup walks
    const int from = SPLIT ? max(lo, (int)blockIdx.z * per * SPAN) : lo;
    const int upto = SPLIT ? min(min(hi, spans * SPAN), ((int)blockIdx.z + 1) * per * SPAN) : hi;
    if (SPLIT && from >= upto) return;  // the fold knows which spans there are

    // Q^T: lane (row r16, g) holds channels 16c + 4g .. + 3 of its row
    f32x4 qf[DB];
    {
        const float* qrow = q + ((size_t)(at + tok) * nq + head) * D + 4 * g;
#pragma unroll
        for (int c = 0; c < DB; ++c) qf[c] = row_ok ? ld4(qrow + 16 * c) : (f32x4){0.f, 0.f, 0.f, 0.f};
    }

    float m = -INFINITY, l = 0.f;
    f32x4 acc[DB];
#pragma unroll
    for (int b = 0; b < DB; ++b) acc[b] = (f32x4){0.f, 0.f, 0.f, 0.f};

    // operands of one tile of 16 keys: lane (key r16, g) reads channels 16c + 4g .. + 3 of its
    // key; lane (channel r16, g) reads keys kb + 4g .. + 3 of its channel in every block
    // The entry of the block table is asked for a tile before (`ask`): the loads of a wave return in their
    // order, so that asking and waiting for it here would wait for every load before it too.
    const unsigned page_keys = (unsigned)page_size * D;
    const int last_page = (hi - 1) / page_size, last_off = hi - 1 - last_page * page_size;
    struct Place {
        int entry, off;
    };
    auto ask_keys = [&](const Walk& w) -> Place {  // beyond the cache: any real key, masked below
        return {table[w.key < hi ? w.page : last_page], w.key < hi ? w.off : last_off};
    };
    auto ask_values = [&](const Walk& w) -> Place {
        return {table[w.key < hi ? w.page : last_page], w.key < hi ? w.off : last_off & ~3};
    };
    auto load_keys = [&](const Place& at_, f32x4 (&f)[DB]) {
        const float* krow = k_cache + (size_t)((unsigned)at_.entry * nkv + hk) * page_keys + at_.off * D + 4 * g;
#pragma unroll
        for (int c = 0; c < DB; ++c) f[c] = ld4(krow + 16 * c);
    };
    auto load_values = [&](const Place& at_, f32x4 (&f)[DB]) {
        const float* vrow = v_cache + (size_t)((unsigned)at_.entry * nkv + hk) * page_keys + r16 * page_size + at_.off;
#pragma unroll
        for (int b = 0; b < DB; ++b) f[b] = ld4(vrow + (size_t)16 * b * page_size);
    };

    // S^T = K Q^T of one tile, the chunks dealt to four accumulators that are added at the
    // end (one chain of dependent instructions would leave the matrix core idle)
    auto scores = [&](const f32x4 (&f)[DB]) -> f32x4 {
        f32x4 part[4];
#pragma unroll
        for (int a4 = 0; a4 < 4; ++a4) part[a4] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int c = 0; c < DB; ++c)
#pragma unroll
            for (int j = 0; j < 4; ++j)
                part[c & 3] =
                    __builtin_amdgcn_mfma_f32_16x16x4f32(f[c][j], qf[c][j], part[c & 3], 0, 0, 0);
        return (part[0] + part[1]) + (part[2] + part[3]);
    };

    // Softmax and second product of the tile at kb, given its scores and its values.  Tiles that every row sees whole,
    // which are most, take no masks.
    const int whole_from = window > 0 ? last_pos - window + 1 : 0;
    auto whole = [&](int kb) { return kb >= whole_from && kb + 15 <= first_pos; };
    auto finish_tile = [&](int kb, f32x4 s, f32x4 (&vals)[DB]) {
#pragma clang fp contract(off)  // a score is rounded before the maximum is subtracted, in every kernel alike
        const bool all = whole(kb);
#pragma unroll
        for (int i = 0; i < 4; ++i) s[i] *= scale;
        if (!all) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int key = kb + 4 * g + i;  // this lane's keys of its own row
                if (!row_ok || key < kstart || key >= kend) s[i] = -INFINITY;
            }
        }
        const float m_new = fmaxf(m, row_max(fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3]))));
        const bool none = m_new == -INFINITY;  // no visible key so far and none here: nothing changes
        const float alpha = none ? 1.f : expf(m - m_new);  // m = -inf before the row's first key: 0
        f32x4 p;
#pragma unroll
        for (int i = 0; i < 4; ++i) p[i] = none ? 0.f : expf(s[i] - m_new);  // masked: exactly 0
        l = fmaf(l, alpha, row_sum((p[0] + p[1]) + (p[2] + p[3])));
        m = m_new;
#pragma unroll
        for (int b = 0; b < DB; ++b)
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[b][i] *= alpha;
        if (!all) {
            // keys no row of the tile sees (beyond the cache, or before the window, whose
            // pages may have been given back) may hold anything: 0 * it must be 0
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int key = kb + 4 * g + i;
                if (key >= hi || key < first_key) {
#pragma unroll
                    for (int b = 0; b < DB; ++b) vals[b][i] = 0.f;
                }
            }
        }
        // ---- O^T += V^T P^T (two chains of dependent instructions in turn) ---------------------
#pragma unroll
        for (int b = 0; b < DB; b += 2)
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int u = b; u < b + 2 && u < DB; ++u)
                    acc[u] = __builtin_amdgcn_mfma_f32_16x16x4f32(vals[u][j], p[j], acc[u], 0, 0, 0);
    };

    // a span is over: its state joins the wave's (a launch that walks whole contexts), or goes to memory
    float m_all = -INFINITY, l_all = 0.f;
    f32x4 acc_all[DB];
    if (!SPLIT) {
#pragma unroll
        for (int b = 0; b < DB; ++b) acc_all[b] = (f32x4){0.f, 0.f, 0.f, 0.f};
    }
    int span = from / SPAN;
    auto finish_span = [&]() {
        if (SPLIT) {
            if (row_ok && r16 < held) {
                float* to = states + ((((size_t)tile * nkv + hk) * spans + span) * AW + wave) * wave_states(held) + r16 * STATE;
#pragma unroll
                for (int b = 0; b < DB; ++b)
#pragma unroll
                    for (int i = 0; i < 4; ++i) to[16 * b + 4 * g + i] = acc[b][i];
                if (g == 0) {
                    to[D] = m;
                    to[D + 1] = l;
                }
            }
            ++span;
        } else {
            const Fold f = fold_of(m_all, m);
            l_all = fold_sum(l_all, l, f);
            m_all = f.m;
#pragma unroll
            for (int b = 0; b < DB; ++b)
#pragma unroll
                for (int i = 0; i < 4; ++i) acc_all[b][i] = fold_sum(acc_all[b][i], acc[b][i], f);
        }
        m = -INFINITY;
        l = 0.f;
#pragma unroll
        for (int b = 0; b < DB; ++b) acc[b] = (f32x4){0.f, 0.f, 0.f, 0.f};
    };

    // Software pipeline over the wave's tiles: the scores of the next tile have been multiplied when a tile
    // is finished, and the keys of the one after travel meanwhile; a tile's values travel while the scores
    // of the next are multiplied.  Inside the loop the loads are issued without a condition and stay where they
    // are written (behind a condition the compiler counts a load as absent and makes every older operand wait
    // for it; left to itself the scheduler moves loads down to their use): the last tiles ask for the last
    // keys again.
    constexpr int STEP = 16 * AW;
    const int mine = from + 16 * ((wave - from / 16) & (AW - 1));  // first tile >= from with index % AW == wave
    if (SPLIT && mine < upto && mine / SPAN > span) finish_span();  // no tile of this wave in the first span
    if (mine < upto) {
        int left = (upto - mine + STEP - 1) / STEP;  // tiles of this wave, the current one included
        int kb = mine;
        const int step_pages = STEP / page_size, step_offs = STEP - step_pages * page_size;
        Walk kw, vw;
        kw.key = kb + r16, kw.page = kw.key / page_size, kw.off = kw.key - kw.page * page_size;
        vw.key = kb + 4 * g, vw.page = vw.key / page_size, vw.off = vw.key - vw.page * page_size;
        f32x4 keys[DB], vals[DB], s_next;
        Place k_next = ask_keys(kw), v_next = ask_values(vw);
        load_keys(k_next, keys);
        load_values(v_next, vals);
        kw.step(STEP, step_pages, step_offs, page_size);
        vw.step(STEP, step_pages, step_offs, page_size);
        k_next = ask_keys(kw);
        v_next = ask_values(vw);
        f32x4 sc = scores(keys);
        if (left > 1) load_keys(k_next, keys);
        kw.step(STEP, step_pages, step_offs, page_size);
        k_next = ask_keys(kw);
        while (--left > 0) {
            s_next = scores(keys);
            kw.step(STEP, step_pages, step_offs, page_size);
            vw.step(STEP, step_pages, step_offs, page_size);
            const Place k_ask = ask_keys(kw), v_ask = ask_values(vw);
            load_keys(k_next, keys);
            __builtin_amdgcn_sched_barrier(0);
            finish_tile(kb, sc, vals);
            load_values(v_next, vals);
            __builtin_amdgcn_sched_barrier(0);
            k_next = k_ask;
            v_next = v_ask;
            sc = s_next;
            kb += STEP;
            if (kb % SPAN < STEP) finish_span();
        }
        finish_tile(kb, sc, vals);
    }
    if (SPLIT) {
        // the last span, and one that holds no tile of this wave
        while (span <= (upto - 1) / SPAN) finish_span();
        return;
    }
    finish_span();
    // ---- fold the waves' states in their order (a wave without visible keys has m = -inf,
    // l = 0 and zero sums: it changes nothing, exactly) ----------------------------------------
    if (wave > 0) {
        fold_ml[wave - 1][0][lane] = m_all;
        fold_ml[wave - 1][1][lane] = l_all;
#pragma unroll
        for (int b = 0; b < DB; ++b) fold_acc[wave - 1][b][lane] = acc_all[b];
    }
    __syncthreads();
    if (wave > 0) return;
#pragma unroll
    for (int w = 0; w < AW - 1; ++w) {
        const Fold f = fold_of(m_all, fold_ml[w][0][lane]);
        l_all = fold_sum(l_all, fold_ml[w][1][lane], f);
        m_all = f.m;
#pragma unroll
        for (int b = 0; b < DB; ++b) {
            const f32x4 other = fold_acc[w][b][lane];
#pragma unroll
            for (int i = 0; i < 4; ++i) acc_all[b][i] = fold_sum(acc_all[b][i], other[i], f);
        }
    }
    if (!row_ok) return;
    // acc_all[b][i] is channel 16b + 4g + i of the lane's row
    float* orow = out + ((size_t)(at + tok) * nq + head) * D + 4 * g;
    const float inv = 1.f / l_all;
#pragma unroll
    for (int b = 0; b < DB; ++b)
        *reinterpret_cast<f32x4*>(orow + 16 * b) = (f32x4){acc_all[b][0] * inv, acc_all[b][1] * inv,
                                                           acc_all[b][2] * inv, acc_all[b][3] * inv};
}

// The states of a split launch folded as the other launch folds them: a workgroup per (tile, kv head),
// 16 lanes a row, D / 16 channels a lane.  Bound by the chain of its loads: a quarter of the threads
// folds the spans of one wave of the launch before (all four in turn took 14 us at nine spans), the first
// quarter then folds the waves.
__global__ __launch_bounds__(256 * AW) void attn_f32_fold_kernel(const float* __restrict__ states, float* __restrict__ out,
                                                                 const int* __restrict__ tile_info,
                                                                 const int* __restrict__ positions, int spans, int held,
                                                                 int nq, int nkv, int window) {
    __shared__ float part_ml[AW][2][256];
    __shared__ float part_acc[AW][DB][256];
    const int tile = blockIdx.x, hk = blockIdx.y;
    const int G = nq / nkv;
    const int at = tile_info[3 * tile], n = tile_info[3 * tile + 1], row0 = tile_info[3 * tile + 2];
    const int rows = n * G;
    const int w = threadIdx.x >> 8, thread = threadIdx.x & 255;
    const int r16 = thread >> 4, part = thread & 15;
    const int row = row0 + r16;
    const bool row_ok = row < rows && r16 < held;
    const int start = positions[at];
    const int first_pos = start + row0 / G;
    const int last_pos = start + (min(rows, row0 + 16) - 1) / G;
    const int first_key = (window > 0 && first_pos - window + 1 > 0) ? first_pos - window + 1 : 0;
    const int s_lo = first_key / SPAN, s_hi = min(last_pos / SPAN + 1, spans);  // the spans that were walked

    float m = -INFINITY, l = 0.f, acc[DB];
#pragma unroll
    for (int b = 0; b < DB; ++b) acc[b] = 0.f;
    if (row_ok) {
#pragma unroll 4
        for (int s = s_lo; s < s_hi; ++s) {
            const float* from = states + ((((size_t)tile * nkv + hk) * spans + s) * AW + w) * wave_states(held) + r16 * STATE;
            const Fold f = fold_of(m, from[D]);
            l = fold_sum(l, from[D + 1], f);
            m = f.m;
#pragma unroll
            for (int b = 0; b < DB; ++b) acc[b] = fold_sum(acc[b], from[16 * b + part], f);
        }
        part_ml[w][0][thread] = m;
        part_ml[w][1][thread] = l;
#pragma unroll
        for (int b = 0; b < DB; ++b) part_acc[w][b][thread] = acc[b];
    }
    __syncthreads();
    if (w > 0 || !row_ok) return;
#pragma unroll
    for (int v = 1; v < AW; ++v) {
        const Fold f = fold_of(m, part_ml[v][0][thread]);
        l = fold_sum(l, part_ml[v][1][thread], f);
        m = f.m;
#pragma unroll
        for (int b = 0; b < DB; ++b) acc[b] = fold_sum(acc[b], part_acc[v][b][thread], f);
    }
    float* orow = out + ((size_t)(at + row / G) * nq + hk * G + row % G) * D;
    const float inv = 1.f / l;
#pragma unroll
    for (int b = 0; b < DB; ++b) orow[16 * b + part] = acc[b] * inv;
}

}  // namespace f32attn

// Every token of the step, single tokens and portions alike.  page_size must be a multiple
// of 4 (the four keys of a lane lie in one page).  `spans` > 0 gives every span of keys to workgroups of
// its own, with `states` [tiles, nkv, spans, 4, held rows of D + 2 in whole lines]; it must cover the longest context.
// `per`: spans a workgroup takes; `held`: rows that the fullest tile has (16 at most).
extern "C" int rl_attn_f32(const float* q, const float* k_cache, const float* v_cache, float* out, float* states,
                           const int* tile_info, int num_tiles, const int* positions,
                           const int* token_slot, const int* block_table, int table_stride,
                           int page_size, int nq, int nkv, int window, float scale, int spans, int per,
                           int held, hipStream_t stream) {
    using namespace f32attn;
    if (num_tiles <= 0) return RL_OK;
    if (nkv < 1 || nq % nkv || page_size < 4 || page_size % 4 || nkv > 65535) return RL_ERR_ARG;
    if (spans < 0 || spans > 65535 || per < 1 || held < 1 || held > 16 || (spans && !states)) return RL_ERR_ARG;
    const dim3 block(AW * RL_WAVE);
    if (!spans) {
        if ((long long)num_tiles * nkv > 0xffffffffll / (AW * RL_WAVE)) return RL_ERR_ARG;
        hipLaunchKernelGGL(attn_f32_kernel<false>, dim3(num_tiles * nkv), block, 0, stream, q, k_cache, v_cache, out,
                           states, tile_info, positions, token_slot, block_table, table_stride, page_size, nq, nkv,
                           window, scale, 0, 1, held);
        return rl_launch_status();
    }
    hipLaunchKernelGGL(attn_f32_kernel<true>, dim3(num_tiles, nkv, (spans + per - 1) / per), block, 0, stream, q, k_cache,
                       v_cache, out, states, tile_info, positions, token_slot, block_table, table_stride, page_size, nq,
                       nkv, window, scale, spans, per, held);
    if (int code = rl_launch_status()) return code;
    hipLaunchKernelGGL(attn_f32_fold_kernel, dim3(num_tiles, nkv), dim3(256 * AW), 0, stream, states, out, tile_info,
                       positions, spans, held, nq, nkv, window);
    return rl_launch_status();
}

extern "C" int rl_attn_f32_span() { return f32attn::SPAN; }
