// bfloat16 product for some hundred rows (prompt steps): out[M,N] = X[M,K] * W[N,K]^T, float32 accumulation on the matrix
// cores; stored as bfloat16, with silu(gate) * up of the packed [gate | up] matrix in the epilogue, or as float32 runs of K.
//
// What bounds it: at these sizes a unit has one tile of 64 to 128 rows on a side, and LDS delivers that tile's operands more
// slowly than the matrix cores take them.  With eight waves beside each other on one tile every operand is read by two and by
// four of them; here four waves share a tile two by two and the other four hold the same tile over the other half of K:
// a chunk's operands are read by two waves each, 3 (WT + XT) cycles of LDS a chunk of 64 k (their way in included) where eight
// waves side by side take 5 WT + 3 XT.
//   * The two groups take the chunks in turn, the even ones and the odd ones: while one multiplies, the other reads its next
//     operands.  A barrier ends each turn, the second group begins one turn later.
//   * The reading group asks memory for a whole chunk, straight into LDS, as many turns ahead as there are buffers.  Nothing
//     waits for all loads: the counter says which are the newest that may still be missing.
//   * No bank is met twice: a row's eight 16-byte units are permuted by the row.
//   * At the end each group takes half of the rows of X: the other group's sums come through the LDS that held the chunks.
#include "common.h"
#include "silu.h"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef u32 u32x2 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) void* rl_lds_ptr;

#define PAIR_LDS (160 * 1024)

struct PairArgs {
    const bf16_t* X;
    const bf16_t* W;
    void* out;
    int M, N, K, ldx, ldw, ldo;
    int tiles_w, tiles_x, splits, k_tiles;  // k_tiles: chunks of 64 k a split
};

// Operand reads from LDS: `at` + T * 2048 holds tile T's first half of the chunk for this lane, `at` ^ 64 the second.  The wait
// stands in the block that asks.
template <int T>
__device__ __forceinline__ void read_tiles(bf16x8 (&f)[T][2], u32 a0, u32 a1) {
    static_assert(T == 2 || T == 3 || T == 4, "tiles of a wave on a side");
    if constexpr (T == 2)
        asm volatile(
            "ds_read_b128 %0, %4\n ds_read_b128 %1, %5\n ds_read_b128 %2, %4 offset:2048\n ds_read_b128 %3, %5 offset:2048\n"
            "s_waitcnt lgkmcnt(0)"
            : "=&v"(f[0][0]), "=&v"(f[0][1]), "=&v"(f[1][0]), "=&v"(f[1][1])
            : "v"(a0), "v"(a1)
            : "memory");
    if constexpr (T == 3)
        asm volatile(
            "ds_read_b128 %0, %6\n ds_read_b128 %1, %7\n ds_read_b128 %2, %6 offset:2048\n ds_read_b128 %3, %7 offset:2048\n"
            "ds_read_b128 %4, %6 offset:4096\n ds_read_b128 %5, %7 offset:4096\n"
            "s_waitcnt lgkmcnt(0)"
            : "=&v"(f[0][0]), "=&v"(f[0][1]), "=&v"(f[1][0]), "=&v"(f[1][1]), "=&v"(f[2][0]), "=&v"(f[2][1])
            : "v"(a0), "v"(a1)
            : "memory");
    if constexpr (T == 4)
        asm volatile(
            "ds_read_b128 %0, %8\n ds_read_b128 %1, %9\n ds_read_b128 %2, %8 offset:2048\n ds_read_b128 %3, %9 offset:2048\n"
            "ds_read_b128 %4, %8 offset:4096\n ds_read_b128 %5, %9 offset:4096\n ds_read_b128 %6, %8 offset:6144\n ds_read_b128 %7, %9 offset:6144\n"
            "s_waitcnt lgkmcnt(0)"
            : "=&v"(f[0][0]), "=&v"(f[0][1]), "=&v"(f[1][0]), "=&v"(f[1][1]), "=&v"(f[2][0]), "=&v"(f[2][1]), "=&v"(f[3][0]), "=&v"(f[3][1])
            : "v"(a0), "v"(a1)
            : "memory");
}

enum PairOut { PAIR_RUNS = 1, PAIR_GLU = 2, PAIR_PLAIN = 3 };

// TW x TX tiles of 16 a wave: a workgroup's tile is 32 TW weight rows x 32 TX rows of X.
template <int TW, int TX, PairOut OUT>
__global__ __launch_bounds__(512) void gemm_pair_kernel(PairArgs a) {
#if defined(__HIP_DEVICE_COMPILE__)  // (the host pass does not know the LDS loads)
    constexpr int WT = 32 * TW, XT = 32 * TX, CHUNK = (WT + XT) * 128;
    constexpr int FIT = PAIR_LDS / CHUNK, D = FIT < 8 ? FIT : 8;  // buffers, and the turns a chunk is asked for ahead
    constexpr int LW = WT / 32, LX = XT / 32, L = LW + LX;        // loads of a wave of the asking group a chunk
    constexpr bool ODD = D % 2 == 1;  // a chunk's askers are its readers
    constexpr int LATER = ((D - (ODD ? 1 : 0)) / 2 - 1) * L;      // of the waves' newest loads, those that may be missing
    constexpr bool GLU = OUT == PAIR_GLU;
    static_assert(D >= 3 && LATER <= 63 && TX % 2 == 0 && (!GLU || TW % 2 == 0), "what the turns below assume");
    __shared__ __attribute__((aligned(1024))) unsigned char lds[D * CHUNK];
    static_assert(sizeof(lds) >= 8 * TW * (TX / 2) * 1024, "half of both groups' sums fit where the chunks were");

    const int tid = threadIdx.x, lane = tid & (RL_WAVE - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid / RL_WAVE);
    const int grp = wave >> 2, w4 = wave & 3, wi = w4 >> 1, xi = w4 & 1;
    const int r16 = lane & 15, g = lane >> 4;

    // the workgroup's tile and split, dealt to the chip's dies as in the many-row product: a die gets a contiguous share, in
    // groups of eight tiles of X walked weight tile by weight tile
    const int tiles = a.tiles_w * a.tiles_x;
    const int split = blockIdx.x / tiles;
    int v = blockIdx.x - split * tiles;
    {
        const int first = split * tiles, die = blockIdx.x & 7, d0 = first & 7;
        const int q = tiles >> 3, r = tiles & 7, d = (die - d0) & 7;
        v = d * q + min(d, r) + (v - d) / 8;
    }
    constexpr int COLS = GLU ? WT / 2 : WT;  // result columns of a tile
    const int per = 8 * a.tiles_w, band = v / per, in = v - band * per;
    const int wide = min(8, a.tiles_x - 8 * band), tw = in / wide;
    const int n0 = tw * COLS, m0 = (8 * band + in - tw * wide) * XT;
    const int k_lo = split * a.k_tiles, k_hi = min(a.K / 64, k_lo + a.k_tiles);

    // Which weight row row r of the tile is.  A wave's (r / (WT / 2)) tiles of 16 go in pairs: plain, a lane's four results of
    // both tiles are eight neighbouring columns; gated, a pair is the gate and up rows of the same columns.  A last tile
    // without a partner has four columns a lane.
    auto weight_row = [&](int r) {
        const int w = r / (WT / 2), t = r % (WT / 2) >> 4, i = r & 15;
        if (GLU) return (t & 1) * a.N + w * (WT / 4) + 16 * (t >> 1) + i;
        const int col = (t | 1) < TW ? 32 * (t >> 1) + 8 * (i >> 2) + 4 * (t & 1) + (i & 3) : 16 * t + i;
        return w * (WT / 2) + col;
    };
    // A load lays a wave's 64 x 16 bytes side by side: eight rows of the tile, unit u of row r at u ^ (r / 2) % 8.
    u32 off[L];
#pragma unroll
    for (int i = 0; i < L; ++i) {
        const int r = 8 * (4 * i + w4) + (lane >> 3);  // rows of W, then of X
        const u32 unit = ((lane & 7) ^ ((r >> 1) & 7)) * 16;
        off[i] = i < LW ? (u32)weight_row(r) * (u32)a.ldw * 2 + unit : (u32)(r - WT) * (u32)a.ldx * 2 + unit;
    }
    const u32 wbytes = (u32)(GLU ? 2 * a.N : a.N) * (u32)a.ldw * 2, xbytes = (u32)a.M * (u32)a.ldx * 2;
    // behind the last chunk the loads find no records and write zeros
    auto ask = [&](int k, u32 at) {
        const u32 offw = (u32)n0 * (u32)a.ldw * 2 + (u32)k * 128, offx = (u32)m0 * (u32)a.ldx * 2 + (u32)k * 128;
        auto rw = __builtin_amdgcn_make_buffer_rsrc((void*)((const char*)a.W + offw), 0, k < k_hi ? wbytes - offw : 0u, 0x00020000);
        auto rx = __builtin_amdgcn_make_buffer_rsrc((void*)((const char*)a.X + offx), 0, k < k_hi ? xbytes - offx : 0u, 0x00020000);
#pragma unroll
        for (int i = 0; i < L; ++i)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(i < LW ? rw : rx, (rl_lds_ptr)(lds + at + (4 * i + w4) * 1024), 16, off[i], 0, 0, 0);
    };
    auto turn = [&]() {
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
    };

    const u32 l0 = (u32)(uintptr_t)(rl_lds_ptr)lds;
    const u32 pos0 = ((u32)g ^ (r16 >> 1)) * 16;
    const u32 w_at = l0 + (u32)(wi * (WT / 2) + r16) * 128 + pos0;
    const u32 x_at = l0 + (u32)(WT + xi * (XT / 2) + r16) * 128 + pos0;

    f32x4 acc[TW][TX];
#pragma unroll
    for (int t = 0; t < TW; ++t)
#pragma unroll
        for (int x = 0; x < TX; ++x) acc[t][x] = (f32x4){0.f, 0.f, 0.f, 0.f};
    bf16x8 wf[TW][2], xf[TX][2];

    // Chunk c is read in turn c - 1 and multiplied in turn c by group c % 2; in turn t the group that reads asks for chunk
    // t + D, into the buffer of chunk t, which has been read.  A turn ends when its waves have waited for what is read next:
    // with an odd D a group's own chunk, behind its products; else the other group's, behind its reads.
    const int chunks = (k_hi - k_lo + 1) & ~1;
#pragma unroll
    for (int c = 0; c < D - 1; ++c)
        if (((c - D + 1) & 1) == grp) ask(k_lo + c, c * CHUNK);
    if (((1 - D) & 1) == grp) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LATER) : "memory");
    turn();
    if (grp) {
        if constexpr (ODD) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LATER) : "memory");
        turn();
    }
    u32 rd = grp * CHUNK, ld = grp ? 0 : (D - 1) * CHUNK;  // chunk c's buffer, and chunk c - 1's
#pragma unroll 1
    for (int c = grp; c < chunks; c += 2) {
        ask(k_lo + c - 1 + D, ld);
        read_tiles<TW>(wf, w_at + rd, (w_at + rd) ^ 64);
        read_tiles<TX>(xf, x_at + rd, (x_at + rd) ^ 64);
        if constexpr (!ODD) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LATER) : "memory");
        turn();
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int t = 0; t < TW; ++t)
#pragma unroll
                for (int x = 0; x < TX; ++x)
                    acc[t][x] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[t][h], xf[x][h], acc[t][x], 0, 0, 0);
        __builtin_amdgcn_s_setprio(0);
        if constexpr (ODD) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LATER) : "memory");
        turn();
        rd += 2 * CHUNK;
        ld += 2 * CHUNK;
        if (rd >= D * CHUNK) rd -= D * CHUNK;
        if (ld >= D * CHUNK) ld -= D * CHUNK;
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // nothing may still be on its way into LDS
    if (!grp) __builtin_amdgcn_s_barrier();
    turn();  // every wave's loads have come

    // group 0 keeps the first half of its wave's rows of X, group 1 the second: the sums in element order, a KB each
    constexpr int HX = TX / 2;
    if (grp) {
#pragma unroll
        for (int t = 0; t < TW; ++t)
#pragma unroll
            for (int x = 0; x < HX; ++x) {
                const f32x4 s = acc[t][x];
                acc[t][x] = acc[t][x + HX];
                acc[t][x + HX] = s;
            }
    }
    f32x4* const handed = reinterpret_cast<f32x4*>(lds);
#pragma unroll
    for (int t = 0; t < TW; ++t)
#pragma unroll
        for (int x = 0; x < HX; ++x) handed[((wave * TW + t) * HX + x) * RL_WAVE + lane] = acc[t][x + HX];
    __syncthreads();
#pragma unroll
    for (int t = 0; t < TW; ++t)
#pragma unroll
        for (int x = 0; x < HX; ++x) acc[t][x] += handed[(((wave ^ 4) * TW + t) * HX + x) * RL_WAVE + lane];

    // ---- results: acc[t][x][i], row m0 + XT / 2 xi + 16 (x + HX grp) + r16 of X ----------------------------
    const u32 elem = OUT == PAIR_RUNS ? 4 : 2;
    char* base = (char*)a.out + ((OUT != PAIR_RUNS ? 0 : (size_t)split * a.M * a.ldo) + (size_t)m0 * a.ldo + n0) * elem;
    const int rows = min(XT, a.M - m0), cols = a.N - n0;
    auto rs = __builtin_amdgcn_make_buffer_rsrc(base, 0, (u32)rows * (u32)a.ldo * elem, 0x00020000);
    bool beyond = false;  // some number of the wave is not below SILU_WIDE
    if constexpr (GLU) {
        // The activation reads its operands rounded to bfloat16, as where the product's result is stored first, and has the
        // many-row product's form, more exact than g / (1 + expf(-g)) * u and shorter: microseconds, that form first, 3,072 x 1,024
        // at 64 / 256 rows 8.7 / 8.6, 11.3 / 10.9, 6,144 x 2,048 at 128 21.4 / 21.0.
        u16x2 most = {0, 0};
#pragma unroll
        for (int t = 0; t < TW; ++t)
#pragma unroll
            for (int x = 0; x < HX; ++x) acc[t][x] = rounded(acc[t][x], most);
        beyond = __any(max(most[0], most[1]) >= SILU_WIDE_BITS);
    }
    // rows and columns that do not exist fall off the records
#pragma unroll
    for (int x = 0; x < HX; ++x) {
        const int row = XT / 2 * xi + 16 * (x + HX * grp) + r16;
#pragma unroll
        for (int t = 0; t < TW; t += 2) {
            const bool two = t + 1 < TW;
            const int t1 = two ? t + 1 : t;
            if constexpr (GLU) {
                const int col = WT / 4 * wi + 8 * t + 4 * g;
                bf16x4 o;
                if (__builtin_expect(beyond, 0)) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) o[i] = (__bf16)silu_times_any(acc[t][x][i], acc[t1][x][i]);
                } else {
#pragma unroll
                    for (int i = 0; i < 4; ++i) o[i] = (__bf16)silu_times(acc[t][x][i], acc[t1][x][i]);
                }
                const bool ok = row < rows && col < cols;
                __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, o), rs, ok ? (row * a.ldo + col) * 2 : -1, 0, 0);
            } else {
                const int col = WT / 2 * wi + (two ? 16 * t + 8 * g : 16 * t + 4 * g);
                const bool ok = row < rows && col < cols;
                if constexpr (OUT == PAIR_PLAIN) {
                    bf16x8 o;
#pragma unroll
                    for (int i = 0; i < 4; ++i) o[i] = (__bf16)acc[t][x][i], o[4 + i] = (__bf16)acc[t1][x][i];
                    if (two)
                        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, o), rs, ok ? (row * a.ldo + col) * 2 : -1, 0, 0);
                    else
                        __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, __builtin_shufflevector(o, o, 0, 1, 2, 3)), rs,
                                                              ok ? (row * a.ldo + col) * 2 : -1, 0, 0);
                } else {
                    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, acc[t][x]), rs, ok ? (row * a.ldo + col) * 4 : -1, 0, 0);
                    if (two)
                        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, acc[t1][x]), rs, ok ? (row * a.ldo + col + 4) * 4 : -1, 0, 0);
                }
            }
        }
    }
#endif
}

template <int TW, int TX>
static int launch_pair(const PairArgs& a, int kind, hipStream_t stream) {
    dim3 grid(a.tiles_w * a.tiles_x * a.splits), block(512);
    if (kind == PAIR_PLAIN)
        hipLaunchKernelGGL((gemm_pair_kernel<TW, TX, PAIR_PLAIN>), grid, block, 0, stream, a);
    else if (kind == PAIR_RUNS)
        hipLaunchKernelGGL((gemm_pair_kernel<TW, TX, PAIR_RUNS>), grid, block, 0, stream, a);
    else if constexpr (TW % 2 == 0 && TW * TX < 16)  // (gated tiles of 128 x 128 are slower than the many-row product's)
        hipLaunchKernelGGL((gemm_pair_kernel<TW, TX, PAIR_GLU>), grid, block, 0, stream, a);
    else
        return RL_ERR_ARG;
    return rl_launch_status();
}

// kind 1: out float32 [splits, M, N], run r of K's chunks in part r.  Kind 2: W = [gate | up] stacked, [2N, K], out
// bfloat16 [M, N] = silu(gate) * up of the products rounded to bfloat16.  Kind 3: out bfloat16 [M, N].
// tw, tx: a tile is 32 tw weight rows x 32 tx rows of X (kind 2: (2, 2), (2, 4) or (4, 2)).  K a multiple of 64, N of 8.
extern "C" int rl_gemm_pair(const void* X, const void* W, void* out, int M, int N, int K, int ldx, int ldw, int ldo,
                            int kind, int tw, int tx, int splits, hipStream_t stream) {
    if (M <= 0 || N <= 0) return RL_OK;
    if (kind < 1 || kind > 3 || !X || !W || !out || K < 64 || K % 64 || N % 8 || ldx % 8 || ldw % 8 || ldo % 8 || ldx < K ||
        ldw < K || ldo < N || splits < 1 || (splits > 1 && kind != PAIR_RUNS) ||
        ((uintptr_t)X | (uintptr_t)W | (uintptr_t)out) % 16)
        return RL_ERR_ARG;
    // offsets inside a matrix are 32-bit, those of rows beyond it too
    const long long limit = 0x7fffffffll;
    if (((long long)M + 128) * ldx * 2 > limit || ((long long)(kind == PAIR_GLU ? 2 : 1) * N + 256) * ldw * 2 > limit || 128ll * ldo * 4 > limit)
        return RL_ERR_ARG;
    PairArgs a;
    a.X = (const bf16_t*)X, a.W = (const bf16_t*)W, a.out = out;
    a.M = M, a.N = N, a.K = K, a.ldx = ldx, a.ldw = ldw, a.ldo = ldo;
    const int cols = (kind == PAIR_GLU ? 16 : 32) * tw, rows = 32 * tx;
    if (tw < 2 || tw > 4 || (tx != 2 && tx != 4)) return RL_ERR_ARG;
    a.tiles_w = (N + cols - 1) / cols, a.tiles_x = (M + rows - 1) / rows, a.splits = splits;
    const int chunks = K / 64;
    a.k_tiles = (chunks + splits - 1) / splits;
    if ((long long)a.k_tiles * (splits - 1) >= chunks) return RL_ERR_ARG;  // every split holds a chunk
    if ((long long)a.tiles_w * a.tiles_x * splits > limit) return RL_ERR_ARG;
#define RL_PAIR(TWV, TXV) \
    if (tw == TWV && tx == TXV) return launch_pair<TWV, TXV>(a, kind, stream)
    RL_PAIR(4, 4);
    RL_PAIR(3, 4);
    RL_PAIR(2, 4);
    RL_PAIR(4, 2);
    RL_PAIR(3, 2);
    RL_PAIR(2, 2);
#undef RL_PAIR
    return RL_ERR_ARG;
}
