// bfloat16 product for many rows (prompt steps): out[M,N] = X[M,K] * W[N,K]^T, float32 accumulation on
// the matrix cores; stored as bfloat16, with silu(gate) * up of the packed [gate | up] matrix in the epilogue, or as
// float32 runs of K.  (As bfloat16, microseconds alone, operands from memory, the library's first: 2,048 rows of 6,144 x 4,096 84.7 /
// 78.9, of 4,096 x 4,096 64.0 / 58.1; 8,926 of 4,096 x 1,024 82.8 / 81.0, of 1,024 x 3,072 62.0 / 55.4.  Inside a prompt step, where X has
// just been written, the first is 2.0 us faster than the library's and the second level; ops.block_plain_plan has the rest.)
//
// What bounds it: the matrix cores, and with real operands the clock they run at (zeros: 2.05 PFLOP/s at
// 8,192 x 8,192 x 8,192, random numbers: 1.55, 1.9 GHz; the library's kernel 2.26 and 1.62), so everything else is kept
// out of their way:
//   * Eight waves on a compute unit, two a SIMD, in two halves that take turns: while one half multiplies, the other
//     reads its next operands from LDS and asks memory for later ones; a barrier ends each turn.  The second half
//     begins one barrier later, that is all that keeps them apart.  (All eight in step: 1.29 against 1.49 PFLOP/s.)
//   * Operands go from memory straight into LDS, 16 bytes a lane, up to two chunks of 64 k ahead; 160 KB of LDS hold 20
//     pieces of 64 rows x 64 k, one load of the workgroup each.  Nothing waits for all loads: the counter says which
//     are the newest that may still be missing.  Memory's answers are what is left: with every load in L2 the kernel
//     runs 6 to 9% faster.
//   * A turn is as long as it can be: 32 matrix instructions (256 x 256 tiles in two turns a chunk; in four 1.49
//     against 1.54 PFLOP/s; asking for W among the matrix instructions instead of beside the reads 1.53 -> 1.49).
//     v_mfma_f32_32x32x16 in place of 16x16x32: 1.54 -> 1.37.
//   * No bank is met twice: a row's eight 16-byte units are permuted by the row (SQ_LDS_BANK_CONFLICT is 0, a read of
//     1 KB takes 4 cycles).
//   * A wave's results are neighbouring columns (128 to 256 bytes of a row), stored 16 bytes a lane: with 32 and
//     64 bytes a wave 2,048 rows of 24,576 x 4,096 took 294 us, so 289, 8,926 rows of 6,144 x 1,024 119 and 112.
// With one piece of X (49 to 64 rows) the weights' bytes bound it: five chunks, 120 KB, are on their way, and a workgroup
// of 64 columns reads X where the kernel that keeps X in registers has 48 (8B gate and up 52.2 -> 48.1 us at 64 rows).
// A workgroup has one tile.  Workgroups that walk several, with the next tile's loads on their way during the
// epilogue, were slower (2,048 rows of 24,576 x 4,096: 316 us): stores and loads share a counter, in order, so the next
// tile's operands waited for this one's results to reach memory.  A new workgroup does not.
#include "common.h"
#include "silu.h"

#include <type_traits>

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef u32 u32x2 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) void* rl_lds_ptr;

#define BT 512        // threads of a workgroup: eight waves, two on a weight side, four on a side of X
#define SLOTS 20      // pieces of 64 rows x 64 k (8 KB) that LDS holds
#define SLOT_BYTES 8192

struct BlockArgs {
    const bf16_t* X;
    const bf16_t* W;
    void* out;
    int M, N, K, ldx, ldw, ldo;
    int tiles_w, tiles_x, splits, k_tiles;  // k_tiles: chunks of 64 k a split
};

template <int N>
struct Int {
    static constexpr int value = N;
};

// Operand reads from LDS.  The wait stands in the block that asks: the registers are whole when it ends,
// and the compiler, which knows nothing of the pieces that are on their way into other buffers, adds no
// wait for those.  a0, a1: the lane's place of the two halves of a chunk in W's buffer; b0, b1: in X's.
template <int NA, int NX>
__device__ __forceinline__ void read_a(bf16x8 (&w)[NA][2][2], bf16x8 (&x)[NX][2], u32 a0, u32 a1, u32 b0, u32 b1) {
    if constexpr (NA == 2 && NX == 4) {
        asm volatile(
            "ds_read_b128 %0, %16\n ds_read_b128 %1, %17\n"
            "ds_read_b128 %2, %16 offset:2048\n ds_read_b128 %3, %17 offset:2048\n"
            "ds_read_b128 %4, %16 offset:8192\n ds_read_b128 %5, %17 offset:8192\n"
            "ds_read_b128 %6, %16 offset:10240\n ds_read_b128 %7, %17 offset:10240\n"
            "ds_read_b128 %8, %18\n ds_read_b128 %9, %19\n"
            "ds_read_b128 %10, %18 offset:8192\n ds_read_b128 %11, %19 offset:8192\n"
            "ds_read_b128 %12, %18 offset:16384\n ds_read_b128 %13, %19 offset:16384\n"
            "ds_read_b128 %14, %18 offset:24576\n ds_read_b128 %15, %19 offset:24576\n"
            "s_waitcnt lgkmcnt(0)"
            : "=&v"(w[0][0][0]), "=&v"(w[0][0][1]), "=&v"(w[0][1][0]), "=&v"(w[0][1][1]),
              "=&v"(w[1][0][0]), "=&v"(w[1][0][1]), "=&v"(w[1][1][0]), "=&v"(w[1][1][1]),
              "=&v"(x[0][0]), "=&v"(x[0][1]), "=&v"(x[1][0]), "=&v"(x[1][1]),
              "=&v"(x[2][0]), "=&v"(x[2][1]), "=&v"(x[3][0]), "=&v"(x[3][1])
            : "v"(a0), "v"(a1), "v"(b0), "v"(b1)
            : "memory");
    } else if constexpr (NA == 2 && NX == 2) {
        asm volatile(
            "ds_read_b128 %0, %12\n ds_read_b128 %1, %13\n"
            "ds_read_b128 %2, %12 offset:2048\n ds_read_b128 %3, %13 offset:2048\n"
            "ds_read_b128 %4, %12 offset:8192\n ds_read_b128 %5, %13 offset:8192\n"
            "ds_read_b128 %6, %12 offset:10240\n ds_read_b128 %7, %13 offset:10240\n"
            "ds_read_b128 %8, %14\n ds_read_b128 %9, %15\n"
            "ds_read_b128 %10, %14 offset:8192\n ds_read_b128 %11, %15 offset:8192\n"
            "s_waitcnt lgkmcnt(0)"
            : "=&v"(w[0][0][0]), "=&v"(w[0][0][1]), "=&v"(w[0][1][0]), "=&v"(w[0][1][1]),
              "=&v"(w[1][0][0]), "=&v"(w[1][0][1]), "=&v"(w[1][1][0]), "=&v"(w[1][1][1]),
              "=&v"(x[0][0]), "=&v"(x[0][1]), "=&v"(x[1][0]), "=&v"(x[1][1])
            : "v"(a0), "v"(a1), "v"(b0), "v"(b1)
            : "memory");
    } else if constexpr (NA == 3 && NX == 2) {
        asm volatile(
            "ds_read_b128 %0, %16\n ds_read_b128 %1, %17\n"
            "ds_read_b128 %2, %16 offset:2048\n ds_read_b128 %3, %17 offset:2048\n"
            "ds_read_b128 %4, %16 offset:8192\n ds_read_b128 %5, %17 offset:8192\n"
            "ds_read_b128 %6, %16 offset:10240\n ds_read_b128 %7, %17 offset:10240\n"
            "ds_read_b128 %8, %16 offset:16384\n ds_read_b128 %9, %17 offset:16384\n"
            "ds_read_b128 %10, %16 offset:18432\n ds_read_b128 %11, %17 offset:18432\n"
            "ds_read_b128 %12, %18\n ds_read_b128 %13, %19\n"
            "ds_read_b128 %14, %18 offset:8192\n ds_read_b128 %15, %19 offset:8192\n"
            "s_waitcnt lgkmcnt(0)"
            : "=&v"(w[0][0][0]), "=&v"(w[0][0][1]), "=&v"(w[0][1][0]), "=&v"(w[0][1][1]),
              "=&v"(w[1][0][0]), "=&v"(w[1][0][1]), "=&v"(w[1][1][0]), "=&v"(w[1][1][1]),
              "=&v"(w[2][0][0]), "=&v"(w[2][0][1]), "=&v"(w[2][1][0]), "=&v"(w[2][1][1]),
              "=&v"(x[0][0]), "=&v"(x[0][1]), "=&v"(x[1][0]), "=&v"(x[1][1])
            : "v"(a0), "v"(a1), "v"(b0), "v"(b1)
            : "memory");
    } else if constexpr (NA == 4 && NX == 2) {
        asm volatile(
            "ds_read_b128 %0, %20\n ds_read_b128 %1, %21\n"
            "ds_read_b128 %2, %20 offset:2048\n ds_read_b128 %3, %21 offset:2048\n"
            "ds_read_b128 %4, %20 offset:8192\n ds_read_b128 %5, %21 offset:8192\n"
            "ds_read_b128 %6, %20 offset:10240\n ds_read_b128 %7, %21 offset:10240\n"
            "ds_read_b128 %8, %20 offset:16384\n ds_read_b128 %9, %21 offset:16384\n"
            "ds_read_b128 %10, %20 offset:18432\n ds_read_b128 %11, %21 offset:18432\n"
            "ds_read_b128 %12, %20 offset:24576\n ds_read_b128 %13, %21 offset:24576\n"
            "ds_read_b128 %14, %20 offset:26624\n ds_read_b128 %15, %21 offset:26624\n"
            "ds_read_b128 %16, %22\n ds_read_b128 %17, %23\n"
            "ds_read_b128 %18, %22 offset:8192\n ds_read_b128 %19, %23 offset:8192\n"
            "s_waitcnt lgkmcnt(0)"
            : "=&v"(w[0][0][0]), "=&v"(w[0][0][1]), "=&v"(w[0][1][0]), "=&v"(w[0][1][1]),
              "=&v"(w[1][0][0]), "=&v"(w[1][0][1]), "=&v"(w[1][1][0]), "=&v"(w[1][1][1]),
              "=&v"(w[2][0][0]), "=&v"(w[2][0][1]), "=&v"(w[2][1][0]), "=&v"(w[2][1][1]),
              "=&v"(w[3][0][0]), "=&v"(w[3][0][1]), "=&v"(w[3][1][0]), "=&v"(w[3][1][1]),
              "=&v"(x[0][0]), "=&v"(x[0][1]), "=&v"(x[1][0]), "=&v"(x[1][1])
            : "v"(a0), "v"(a1), "v"(b0), "v"(b1)
            : "memory");
    } else if constexpr (NA == 2 && NX == 1) {
        asm volatile(
            "ds_read_b128 %0, %10\n ds_read_b128 %1, %11\n"
            "ds_read_b128 %2, %10 offset:2048\n ds_read_b128 %3, %11 offset:2048\n"
            "ds_read_b128 %4, %10 offset:8192\n ds_read_b128 %5, %11 offset:8192\n"
            "ds_read_b128 %6, %10 offset:10240\n ds_read_b128 %7, %11 offset:10240\n"
            "ds_read_b128 %8, %12\n ds_read_b128 %9, %13\n"
            "s_waitcnt lgkmcnt(0)"
            : "=&v"(w[0][0][0]), "=&v"(w[0][0][1]), "=&v"(w[0][1][0]), "=&v"(w[0][1][1]),
              "=&v"(w[1][0][0]), "=&v"(w[1][0][1]), "=&v"(w[1][1][0]), "=&v"(w[1][1][1]),
              "=&v"(x[0][0]), "=&v"(x[0][1])
            : "v"(a0), "v"(a1), "v"(b0), "v"(b1)
            : "memory");
    } else {
        static_assert(NX < 0, "no such read");
    }
}
// the pieces of W behind the first NA
template <int NA, int NB>
__device__ __forceinline__ void read_b(bf16x8 (&w)[NA][2][2], u32 a0, u32 a1) {
    if constexpr (NA == 2 && NB == 1) {
        asm volatile(
            "ds_read_b128 %0, %4 offset:16384\n ds_read_b128 %1, %5 offset:16384\n"
            "ds_read_b128 %2, %4 offset:18432\n ds_read_b128 %3, %5 offset:18432\n"
            "s_waitcnt lgkmcnt(0)"
            : "=&v"(w[0][0][0]), "=&v"(w[0][0][1]), "=&v"(w[0][1][0]), "=&v"(w[0][1][1])
            : "v"(a0), "v"(a1)
            : "memory");
    } else if constexpr (NA == 2 && NB == 2) {
        asm volatile(
            "ds_read_b128 %0, %8 offset:16384\n ds_read_b128 %1, %9 offset:16384\n"
            "ds_read_b128 %2, %8 offset:18432\n ds_read_b128 %3, %9 offset:18432\n"
            "ds_read_b128 %4, %8 offset:24576\n ds_read_b128 %5, %9 offset:24576\n"
            "ds_read_b128 %6, %8 offset:26624\n ds_read_b128 %7, %9 offset:26624\n"
            "s_waitcnt lgkmcnt(0)"
            : "=&v"(w[0][0][0]), "=&v"(w[0][0][1]), "=&v"(w[0][1][0]), "=&v"(w[0][1][1]),
              "=&v"(w[1][0][0]), "=&v"(w[1][0][1]), "=&v"(w[1][1][0]), "=&v"(w[1][1][1])
            : "v"(a0), "v"(a1)
            : "memory");
    } else {
        static_assert(NA < 0, "no such read");
    }
}

enum BlockOut { OUT_RUNS = 1, OUT_GLU = 2, OUT_PLAIN = 3 };

// NW x NX pieces of 64 rows: a workgroup's tile is 64 NW weight rows x 64 NX rows of X.
template <int NW, int NX, BlockOut OUT>
__global__ __launch_bounds__(BT) void gemm_block_kernel(BlockArgs a) {
#if defined(__HIP_DEVICE_COMPILE__)  // (the host pass does not know the LDS loads)
    constexpr int U = NW + NX;  // pieces of a chunk
    // Buffers for three chunks and more: a chunk is one phase, its loads D chunks ahead.  For two and a half: W has
    // three buffers (four), X two, and a chunk is two phases, which read W's pieces one half (two) after the other.
    constexpr bool ONE = SLOTS / U >= 3;
    constexpr int NA = ONE ? NW : 2, NB = NW - NA;
    constexpr int XB = ONE ? SLOTS / U : 2, WB = ONE ? XB : (SLOTS - XB * NX) / NW;
    constexpr int D = XB - 1;
    // loads of a thread that may still be on their way when the next chunk has to be there
    constexpr int AHEAD_X = (XB - 1) * U, AHEAD_W = (WB - 1) * NX + (WB - 2) * NW;
    constexpr int AHEAD = ONE ? (D - 1) * U : (AHEAD_X < AHEAD_W ? AHEAD_X : AHEAD_W);
    constexpr bool GLU = OUT == OUT_GLU;
    static_assert(WB * NW + XB * NX <= SLOTS && WB >= 2 && AHEAD <= 63, "the buffers fit, and the counter");
    __shared__ __attribute__((aligned(1024))) unsigned char lds[SLOTS * SLOT_BYTES];
    constexpr u32 WBUF = NW * SLOT_BYTES, XBUF = NX * SLOT_BYTES, X0 = WB * WBUF;

    const int tid = threadIdx.x, lane = tid & (RL_WAVE - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid / RL_WAVE);
    const int wi = wave & 1, xi = wave >> 1;
    const int r16 = lane & 15, g = lane >> 4;

    // ---- the workgroup's tile and split --------------------------------------------------------
    // Workgroups go to the chip's eight dies in turn: a die gets a contiguous share of the tiles, in groups
    // of eight tiles of X walked weight tile by weight tile, so that what its workgroups read at a time is
    // mostly shared in its L2.
    const int tiles = a.tiles_w * a.tiles_x;
    const int split = blockIdx.x / tiles;
    int v = blockIdx.x - split * tiles;
    {
        const int first = split * tiles, die = blockIdx.x & 7, d0 = first & 7;
        const int q = tiles >> 3, r = tiles & 7, d = (die - d0) & 7;  // the split's d-th die
        v = d * q + min(d, r) + (v - d) / 8;
    }
    constexpr int COLS = GLU ? 32 * NW : 64 * NW;  // result columns of a tile
    const int per = 8 * a.tiles_w, grp = v / per, in = v - grp * per;
    const int wide = min(8, a.tiles_x - 8 * grp), tw = in / wide;
    const int n0 = tw * COLS, m0 = (8 * grp + in - tw * wide) * (64 * NX);
    const int k_lo = split * a.k_tiles, k_hi = min(a.K / 64, k_lo + a.k_tiles);

    // ---- the loads --------------------------------------------------------------------------------
    // A load lays a wave's 64 x 16 bytes side by side: rows 8 wave .. + 7 of the piece.  A row's eight
    // 16-byte units are permuted (unit u of row r at u ^ (r / 2) % 8): reads meet every bank once.
    const int lr = 8 * wave + (lane >> 3);
    const u32 lunit = ((lane & 7) ^ ((lr >> 1) & 7)) * 16;
    // Which weight row LDS row lr of piece u holds.  Its wave (lr / 32) has neighbouring columns in all pieces,
    // so that a wave's stores fill whole lines of the result one after another.  Plain: a lane's four results of
    // a piece's two tiles of 16 are eight neighbouring columns.  Gated: the two tiles are the gate and up rows
    // of the same columns, and a lane's four results of two pieces are neighbours.
    auto weight_row = [&](int u) {
        const int w = lr >> 5, t = (lr >> 4) & 1, i = lr & 15;
        if (!GLU) return w * (32 * NW) + 32 * u + 8 * (i >> 2) + 4 * t + (i & 3);
        const int col = (u | 1) < NW ? 16 * (u & ~1) + 8 * (i >> 2) + 4 * (u & 1) + (i & 3) : 16 * u + i;
        return t * a.N + w * (16 * NW) + col;
    };
    u32 woff[NW], xoff[NX];
#pragma unroll
    for (int u = 0; u < NW; ++u) woff[u] = (u32)weight_row(u) * (u32)a.ldw * 2 + lunit;
#pragma unroll
    for (int u = 0; u < NX; ++u) xoff[u] = (u32)(lr + u * 64) * (u32)a.ldx * 2 + lunit;
    const u32 wbytes = (u32)(GLU ? 2 * a.N : a.N) * (u32)a.ldw * 2, xbytes = (u32)a.M * (u32)a.ldx * 2;

    // behind the last chunk the loads find no records and write zeros that nobody reads
    auto load_w = [&](int k, u32 at) {
        const u32 off = (u32)n0 * (u32)a.ldw * 2 + (u32)k * 128;
        auto rs = __builtin_amdgcn_make_buffer_rsrc((void*)((const char*)a.W + off), 0, k < k_hi ? wbytes - off : 0u, 0x00020000);
#pragma unroll
        for (int u = 0; u < NW; ++u)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (rl_lds_ptr)(lds + at + wave * 1024 + u * SLOT_BYTES), 16, woff[u], 0, 0, 0);
    };
    auto load_x = [&](int k, u32 at) {
        const u32 off = (u32)m0 * (u32)a.ldx * 2 + (u32)k * 128;
        auto rs = __builtin_amdgcn_make_buffer_rsrc((void*)((const char*)a.X + off), 0, k < k_hi ? xbytes - off : 0u, 0x00020000);
#pragma unroll
        for (int u = 0; u < NX; ++u)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (rl_lds_ptr)(lds + at + wave * 1024 + u * SLOT_BYTES), 16, xoff[u], 0, 0, 0);
    };

    // ---- operands -------------------------------------------------------------------------------
    const u32 l0 = (u32)(uintptr_t)(rl_lds_ptr)lds;
    const u32 pos0 = ((u32)g ^ ((r16 >> 1) & 7)) * 16;
    const u32 w_at0 = l0 + (u32)(wi * 32 + r16) * 128 + pos0, w_at1 = w_at0 ^ 64;
    const u32 x_at0 = l0 + (u32)(xi * 16 + r16) * 128 + pos0, x_at1 = x_at0 ^ 64;
    u32 rd_w = 0, rd_x = X0;  // the buffers that hold the chunk being multiplied
    f32x4 acc[NW][2][NX];
    bf16x8 wf[NA][2][2], xf[NX][2];

    auto products = [&](auto first_c, auto count_c) {
        constexpr int first = decltype(first_c)::value, count = decltype(count_c)::value;
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int u = 0; u < count; ++u)
#pragma unroll
                for (int t = 0; t < 2; ++t)
#pragma unroll
                    for (int x = 0; x < NX; ++x)
                        acc[first + u][t][x] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[u][t][h], xf[x][h], acc[first + u][t][x], 0, 0, 0);
        __builtin_amdgcn_s_setprio(0);
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
    };
    // in the order in which the loop asks
    if constexpr (ONE) {
#pragma unroll
        for (int t = 0; t < D; ++t) load_w(k_lo + t, t * WBUF), load_x(k_lo + t, X0 + t * XBUF);
    } else {
#pragma unroll
        for (int t = -(WB - 1 > XB ? WB - 1 : XB); t < 0; ++t) {
            if (t >= 1 - WB) load_w(k_lo + t + WB - 1, (t + WB - 1) * WBUF);
            if (t >= -XB) load_x(k_lo + t + XB, X0 + (t + XB) * XBUF);
        }
    }
#pragma unroll
    for (int u = 0; u < NW; ++u)
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int x = 0; x < NX; ++x) acc[u][t][x] = (f32x4){0.f, 0.f, 0.f, 0.f};
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(AHEAD) : "memory");
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    if (wave >= 4) __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);

    u32 ld_w = (WB - 1) * WBUF, ld_x = X0 + (XB - 1) * XBUF;  // the buffers that were multiplied last
#pragma unroll 1
    for (int k = k_lo; k < k_hi; ++k) {
        const u32 a0 = w_at0 + rd_w, a1 = w_at1 + rd_w;
        // the first pieces of W, all of X
        load_w(k + WB - 1, ld_w);
        if constexpr (ONE) load_x(k + D, ld_x);
        read_a<NA, NX>(wf, xf, a0, a1, x_at0 + rd_x, x_at1 + rd_x);
        if constexpr (ONE) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(AHEAD) : "memory");
        products(Int<0>{}, Int<NA>{});
        if constexpr (!ONE) {  // the other pieces of W; X's buffer is free
            load_x(k + XB, rd_x);
            read_b<NA, NB>(wf, a0, a1);
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"(AHEAD) : "memory");
            products(Int<NA>{}, Int<NB>{});
        }
        ld_x = rd_x;
        ld_w = rd_w;
        rd_w = rd_w == (WB - 1) * WBUF ? 0 : rd_w + WBUF;
        rd_x = rd_x == X0 + (XB - 1) * XBUF ? X0 : rd_x + XBUF;
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // nothing may still be on its way into LDS when it is given back
    if (wave < 4) __builtin_amdgcn_s_barrier();
    // ---- results: acc[u][t][x][i], row m0 + 64 x + 16 xi + r16 of X ----------------------------
    const u32 elem = OUT == OUT_RUNS ? 4 : 2;
    char* base = (char*)a.out + ((OUT != OUT_RUNS ? 0 : (size_t)split * a.M * a.ldo) + (size_t)m0 * a.ldo + n0) * elem;
    const int rows = min(64 * NX, a.M - m0), cols = a.N - n0;
    auto rs = __builtin_amdgcn_make_buffer_rsrc(base, 0, (u32)rows * (u32)a.ldo * elem, 0x00020000);
    // rows and columns that do not exist fall off the records
    auto finish = [&](int x, auto any_c) {
        const int row = 64 * x + 16 * xi + r16;
        bf16x8 o;
#pragma unroll
        for (int u = 0; u < NW; ++u) {
            if constexpr (GLU) {
                const bool pair = (u | 1) < NW;
                const int col = 16 * NW * wi + (pair ? 16 * (u & ~1) + 8 * g + 4 * (u & 1) : 16 * u + 4 * g);
                const bool in = row < rows && col < cols;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float gate = acc[u][0][x][i], up = acc[u][1][x][i];
                    o[4 * (u & 1) + i] = (__bf16)(decltype(any_c)::value ? silu_times_any(gate, up) : silu_times(gate, up));
                }
                if (pair && (u & 1))
                    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, o), rs, in ? (row * a.ldo + col - 4) * 2 : -1, 0, 0);
                else if (!pair)
                    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, __builtin_shufflevector(o, o, 0, 1, 2, 3)), rs,
                                                          in ? (row * a.ldo + col) * 2 : -1, 0, 0);
            } else {
                const int col = 32 * NW * wi + 32 * u + 8 * g;
                const bool in = row < rows && col < cols;
                if constexpr (OUT == OUT_PLAIN) {
#pragma unroll
                    for (int i = 0; i < 8; ++i) o[i] = (__bf16)acc[u][i >> 2][x][i & 3];
                    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, o), rs, in ? (row * a.ldo + col) * 2 : -1, 0, 0);
                    continue;
                }
#pragma unroll
                for (int t = 0; t < 2; ++t)
                    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, acc[u][t][x]), rs,
                                                           in ? (row * a.ldo + col + 4 * t) * 4 : -1, 0, 0);
            }
        }
    };
    u16x2 most = {0, 0};
    if constexpr (GLU) {
        // the activation reads its operands rounded to bfloat16, as where the product's result is stored first
#pragma unroll
        for (int x = 0; x < NX; ++x)
#pragma unroll
            for (int u = 0; u < NW; ++u)
#pragma unroll
                for (int t = 0; t < 2; ++t) acc[u][t][x] = rounded(acc[u][t][x], most);
    }
    if (__builtin_expect(!GLU || !__any(max(most[0], most[1]) >= SILU_WIDE_BITS), 1)) {
#pragma unroll
        for (int x = 0; x < NX; ++x) finish(x, Int<0>{});
    } else {
#pragma unroll
        for (int x = 0; x < NX; ++x) finish(x, Int<1>{});
    }
#endif
}

template <int NW, int NX>
static int launch_block(const BlockArgs& a, int kind, hipStream_t stream) {
    dim3 grid(a.tiles_w * a.tiles_x * a.splits), block(BT);
    if (kind == OUT_GLU)
        hipLaunchKernelGGL((gemm_block_kernel<NW, NX, OUT_GLU>), grid, block, 0, stream, a);
    else if (kind == OUT_PLAIN)
        hipLaunchKernelGGL((gemm_block_kernel<NW, NX, OUT_PLAIN>), grid, block, 0, stream, a);
    else
        hipLaunchKernelGGL((gemm_block_kernel<NW, NX, OUT_RUNS>), grid, block, 0, stream, a);
    return rl_launch_status();
}

// kind 1: out float32 [splits, M, N], run r of K's chunks in part r.  Kind 2: W = [gate | up] stacked, [2N, K], out
// bfloat16 [M, N] = silu(gate) * up of the products rounded to bfloat16.  Kind 3: out bfloat16 [M, N].
// nw, nx: pieces of 64 rows of a tile (2 to 4, 2 or 4; 2, 1).  K a multiple of 64, N of 8.
extern "C" int rl_gemm_block(const void* X, const void* W, void* out, int M, int N, int K, int ldx, int ldw, int ldo,
                             int kind, int nw, int nx, int splits, hipStream_t stream) {
    if (M <= 0 || N <= 0) return RL_OK;
    if ((kind != OUT_RUNS && kind != OUT_GLU && kind != OUT_PLAIN) || !X || !W || !out || K < 64 || K % 64 || N % 8 || ldx % 8 || ldw % 8 || ldo % 8 || ldx < K ||
        ldw < K || ldo < N || splits < 1 || (splits > 1 && kind != OUT_RUNS) ||
        ((uintptr_t)X | (uintptr_t)W | (uintptr_t)out) % 16)
        return RL_ERR_ARG;
    // offsets inside a matrix are 32-bit, those of rows beyond it too
    const long long limit = 0x7fffffffll;
    if (((long long)M + 256) * ldx * 2 > limit || ((long long)(kind == OUT_GLU ? 2 : 1) * N + 256) * ldw * 2 > limit || 256ll * ldo * 4 > limit)
        return RL_ERR_ARG;
    BlockArgs a;
    a.X = (const bf16_t*)X, a.W = (const bf16_t*)W, a.out = out;
    a.M = M, a.N = N, a.K = K, a.ldx = ldx, a.ldw = ldw, a.ldo = ldo;
    const int cols = (kind == OUT_GLU ? 32 : 64) * nw, rows = 64 * nx;
    a.tiles_w = (N + cols - 1) / cols, a.tiles_x = (M + rows - 1) / rows, a.splits = splits;
    const int chunks = K / 64;
    a.k_tiles = (chunks + splits - 1) / splits;
    if ((long long)a.k_tiles * (splits - 1) >= chunks) return RL_ERR_ARG;  // every split holds a chunk
    if ((long long)a.tiles_w * a.tiles_x * splits > limit) return RL_ERR_ARG;
#define RL_BLOCK(NWV, NXV) \
    if (nw == NWV && nx == NXV) return launch_block<NWV, NXV>(a, kind, stream)
    RL_BLOCK(4, 4);
    RL_BLOCK(3, 4);
    RL_BLOCK(2, 4);
    RL_BLOCK(4, 2);
    RL_BLOCK(3, 2);
    RL_BLOCK(2, 2);
    RL_BLOCK(2, 1);
#undef RL_BLOCK
    return RL_ERR_ARG;
}
