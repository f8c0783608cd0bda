// Float32 matrix product C[M,N] = A[M,K] * W[N,K]^T on the matrix cores' bfloat16 instruction
// (v_mfma_f32_16x16x32_bf16), without the loss of a bfloat16 product: every float32 operand is
// split into three bfloat16 numbers that add up to it (24 bits of mantissa are 8 + 8 + 8), and a
// product of two operands is the six partial products
//   hi hi + (hi mid + mid hi) + (mid mid + hi lo + lo hi),
// each exact before it is added up in float32.  The three left out come to 2^-24 of the product at
// most, half a unit in its last place (|mid| <= 2^-8, |lo| <= 2^-17 of the operand's power of two: mid lo and
// lo mid are 2^-25 each), and far less on the average.  The float32 instruction (v_mfma_f32_16x16x4_f32) has 157
// TFLOP/s at most, and the kernel on it that this one replaces reached 101; six bfloat16 instructions
// come to a sixth of 2.5 PFLOP/s, of which bfloat16 products of real operands reach 0.6.  Measured at 2,048
// rows: 6,144 x 4,096 1,018 -> 453 us, 24,576 x 4,096 4,259 -> 1,624 us, 4,096 x 12,288 2,007 -> 817 us
// (227 to 254 TFLOP/s); at 225 rows of a small model 6,144 x 1,024 53 -> 36 us and 1,024 x 3,072 68 -> 20
// us (22 and 18 where a wave has a run).  Error against 64 bits over normal operands, relative to the result: K = 4,096 4.1e-7 -> 3.4e-7,
// K = 12,288 7.0e-7 -> 6.0e-7.
//
// One order of summation for every output element, whatever M, the tile it falls in or what
// else is in the batch, so that results are equal bit for bit however the rows are cut:
//   * K is cut in chunks of 32; the chunks are dealt in 8 contiguous runs of ceil(chunks / 8);
//   * a run's chunks are walked in ascending order; a chunk is six matrix instructions on one
//     accumulator, the small partial products first, lane group g supplying k = 8 g .. 8 g + 7;
//   * the 8 runs' results are added in their order.
// The instruction rounds its sums down (a product of 4,096 k came out 0.75e-7 of its size too low on the
// average, the same for every element, which layers add up): odd runs work on -A and are subtracted, so
// that what two neighbouring runs lose cancels.  k beyond K contribute zeros.
//
// The exponents of the pieces: a bfloat16 number ends where float32 does, so the lower pieces of an
// operand below 2^-109 would not exist.  Operands are multiplied by 2^24 before they are split: the
// smallest float32 number, 2^-149, is then the normal number 2^-125, every piece of every operand below
// 2^103 is exact, and the sum times 2^-48 is the result.  What the pieces cannot hold is computed again
// without them: an element that comes out infinite or not a number (an infinite operand meets a zero
// piece of the other; an operand from 2^103 or a result from 2^80 on is infinite once scaled) is
// summed in 64 bits by the vector units instead.
//
// So are sums of up to three k, in a kernel of their own.  What is left out and what the instruction drops of a sum come to 2.6 x 2^-24 of a lone
// product at most, 0.57 x 2^-24 root mean square (a multiply-add: 1.0 and 0.43); the sums of the float32 instruction
// are the further off from four k on (root mean square in 2^-24 of the result, it and this, 200 rows of normal
// operands: 4 k 0.67 / 0.54, 8 0.90 / 0.53, 32 1.32 / 0.63, 128 1.56 / 0.93, 1,024 3.54 / 2.72, 4,096 6.87 / 5.71,
// 12,288 11.8 / 10.0; of positive ones 4 k 0.61 / 0.49, 32 0.91 / 0.59, 4,096 2.02 / 1.64).  Up to 32 k there is one run
// and nothing cancels what the instruction rounds down: 0.15 x 2^-24 of positive operands' result at 4 k, 0.03 at 32.
// A long sum that one product makes up alone, the others being zeros, has that product's error.
//
// The transposed product is computed (W supplies the A operand, the rows of A the B operand),
// so a lane's four results are four consecutive n of one row of C.
#include "common.h"

#include <type_traits>

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

#define FRUNS 8  // runs of K = waves per workgroup of the streaming kernel
#define FCH 32   // k per chunk
#define FEW 3    // k up to which sums are in 64 bits

// Two floats as two bfloat16 side by side (round to nearest even: one instruction), and what
// that leaves of them.
__device__ inline uint32_t take_bf16(float& a, float& b) {
    const bf16x2 h = __builtin_convertvector((f32x2){a, b}, bf16x2);
    const uint32_t u = __builtin_bit_cast(uint32_t, h);
    a -= __builtin_bit_cast(float, u << 16);
    b -= __builtin_bit_cast(float, u & 0xffff0000u);
    return u;
}

struct Split {
    bf16x8 p[3];  // hi, mid, lo of eight consecutive k
};

constexpr float UP = 0x1p24f, DOWN = 0x1p-48f;  // what operands and sums are multiplied by

// `up`: UP, or -UP for A in odd runs
__device__ inline Split split8(f32x4 x, f32x4 y, float up = UP) {
    u32x4 p[3];
    float v[8];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        v[j] = x[j] * up;
        v[4 + j] = y[j] * up;
    }
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) p[i][j] = take_bf16(v[2 * j], v[2 * j + 1]);
    Split s;
#pragma unroll
    for (int i = 0; i < 3; ++i) s.p[i] = __builtin_bit_cast(bf16x8, p[i]);
    return s;
}

// the six partial products of one chunk, the smallest first: piece of W, piece of A
__device__ constexpr int PIECE_W[6] = {2, 0, 1, 1, 0, 0};
__device__ constexpr int PIECE_A[6] = {0, 2, 1, 0, 1, 0};

// An element the pieces could not hold, in 64 bits; 16 operands of each row are asked for together.  (One k a time, an
// infinite operand in each of 256 rows took 4,096 x 4,096 to 14.7 ms; so it is 1.9.)
__device__ inline float wide_sum(const float* a, const float* w, int K) {
    double s = 0.0;
    int k = 0;
    for (; k + 16 <= K && s == s; k += 16) {
        float x[16], y[16];
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            x[j] = a[k + j];
            y[j] = w[k + j];
        }
#pragma unroll
        for (int j = 0; j < 16; ++j) s = fma((double)x[j], (double)y[j], s);
    }
    for (; k < K && s == s; ++k) s = fma((double)a[k], (double)w[k], s);
    return (float)s;
}

// the sum as the element it stands for, or that in 64 bits where the sum is no finite number
__device__ inline float finite_or_wide(float v, const float* a, const float* w, int K) {
    return __builtin_isfinite(v) ? v * DOWN : wide_sum(a, w, K);
}

// GLU: W is a gate and an up matrix, N rows each, one behind the other, and a result is silu(gate) * up of the two
// products.  Sixteen rows of a tile are the gate and up rows of eight columns, two and two in turn, so that a lane's four
// results are two columns' pairs, whatever the tile.  The bits are those of the product and the activation's kernel one after
// the other, which the results, twice as many, went through memory for: microseconds of a step before / with this, 0.6B
// three prompts of 225 tokens 3,602 / 3,457, 8B a prompt of 2,048 140,050 / 138,250, eight requests decode 7,367 / 7,174.
template <bool GLU>
__device__ inline size_t row_of(int slot, int N) {
    if (!GLU) return min(slot, N - 1);
    const int col = (slot >> 4) * 8 + ((slot >> 1) & 6) + (slot & 1);
    return (size_t)min(col, N - 1) + (slot & 2 ? N : 0);
}
__device__ inline float silu_mul(float g, float u) {
    const Glu plain = {0.f, 0.f, 0, nullptr};
    return glu_act(g, u, plain);
}

// 16 bytes from any address of a float: rows may begin anywhere (the hardware asks for 4-byte alignment)
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));
__device__ inline f32x4 load4(const float* p) { return *reinterpret_cast<const f32x4u*>(p); }

// What K is: a multiple of 32 (chunks are WHOLE), of 4 (pieces of four k are there or beyond K), or neither.
enum Length { ELEMENTS, PIECES, WHOLE };

// Four k of a row from p[at] on, zeros beyond K; the row begins `before` elements in front of p.  What lies beyond
// is the row's first elements read for nothing: no load stands behind a condition.  (Where K was not a multiple of
// 32 or a row not aligned, operands were read one checked element at a time: 4,096 x 1,000 took 45 us at 225 rows,
// 99 at 512 and 218 at 2,048, where PIECES take 28, 47 and 106; 4,096 x 333 at 8 rows took 6.9 us and takes 3.8.)
template <Length L>
__device__ inline f32x4 load_k4(const float* p, int at, int before, int K) {
    if (L == WHOLE) return load4(p + at);
    const int left = K - before - at;
    f32x4 v;
    if (L == PIECES) {
        v = load4(p + (left > 0 ? at : -before));
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = left > 0 ? v[i] : 0.f;
        return v;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float x = p[i < left ? at + i : -before];
        v[i] = i < left ? x : 0.f;
    }
    return v;
}

// ---- few rows, or few k: the weights are streamed once ------------------------------------------
// One workgroup per NT tiles of 16 rows of W and MT of A, one wave per run of K.  Bound by the weights' bytes, and from
// a few rows on by the rows of A beside them, which every workgroup reads whole.  With one tile of A up to 16 rows
// (f32_plan says when NT is 2 or 3), with two for 17 to 32 rows over short ones and for any number of rows over at
// most 256 k, where a wave has one chunk and the shared tiles below walk a chain of chunks or leave the runs to a second
// kernel: 17 rows over 6,144 x 1,024 14.6 -> 11.5 us, over 1,024 x 128 6.0 -> 3.3, 225 rows 8.4 -> 4.4.
template <int NT, int MT, bool GLU>
__global__ __launch_bounds__(FRUNS* RL_WAVE) void gemm_f32_stream_kernel(
    const float* __restrict__ A, const float* __restrict__ W, float* __restrict__ C, int M, int N,
    int K, int lda, int ldw, int ldc) {
    __shared__ float red[FRUNS][NT * MT * 256];

    const int lane = threadIdx.x & (RL_WAVE - 1);
    const int wave = threadIdx.x / RL_WAVE;
    const int r16 = lane & 15;
    const int g = lane >> 4;
    const int n0 = blockIdx.x * NT * 16, m0 = blockIdx.y * MT * 16;

    // rows beyond the matrices read the last row; their results are dropped at the end
    const float* wrow[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) wrow[nt] = W + row_of<GLU>(n0 + nt * 16 + r16, N) * ldw + 8 * g;
    const float* arow[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) arow[mt] = A + (size_t)min(m0 + mt * 16 + r16, M - 1) * lda + 8 * g;

    f32x4 acc[NT][MT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) acc[nt][mt] = (f32x4){0.f, 0.f, 0.f, 0.f};

    const int chunks = (K + FCH - 1) / FCH;
    const int per = (chunks + FRUNS - 1) / FRUNS;
    const int c_lo = min(chunks, wave * per), c_hi = min(chunks, c_lo + per);

    // two chunks are asked for together: 256 contiguous bytes of every row (with many tiles one, whose
    // loads are as many)
    constexpr int U = NT + MT > 3 ? 1 : 2;
    struct Rows {
        f32x4 w[U][NT][2], a[U][MT][2];
    };
    auto load_group = [&](int c, Rows& r) {  // whole chunks: no predicate
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
#pragma unroll
                for (int nt = 0; nt < NT; ++nt)
                    r.w[u][nt][h] = load4(wrow[nt] + (c + u) * FCH + 4 * h);
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) r.a[u][mt][h] = load4(arow[mt] + (c + u) * FCH + 4 * h);
            }
        // the loads stay here, in front of the other group's products (left to itself the
        // scheduler moves them down to their use and nothing is in flight during the products)
        __builtin_amdgcn_sched_barrier(0);
    };
    auto products = [&](const f32x4 (&w)[NT][2], const f32x4 (&a)[MT][2]) {
        Split as[MT];
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) as[mt] = split8(a[mt][0], a[mt][1], wave & 1 ? -UP : UP);
        constexpr int NB = NT % 2 ? 1 : 2;  // tiles whose instructions alternate
#pragma unroll
        for (int n0 = 0; n0 < NT; n0 += NB) {
            Split ws[NB];
#pragma unroll
            for (int j = 0; j < NB; ++j) ws[j] = split8(w[n0 + j][0], w[n0 + j][1]);
#pragma unroll
            for (int s = 0; s < 6; ++s)
#pragma unroll
                for (int j = 0; j < NB; ++j)
#pragma unroll
                    for (int mt = 0; mt < MT; ++mt)
                        acc[n0 + j][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                            ws[j].p[PIECE_W[s]], as[mt].p[PIECE_A[s]], acc[n0 + j][mt], 0, 0, 0);
        }
    };
    auto group_products = [&](const Rows& r) {
#pragma unroll
        for (int u = 0; u < U; ++u) products(r.w[u], r.a[u]);
    };
    // Groups of whole chunks go through two sets of registers in turn: the group after next
    // is asked for before this one is multiplied.  Inside the loop no load stands behind a
    // condition (behind one the compiler counts it as absent and makes the oldest operand wait
    // for the newest load); what the loop leaves, and the chunks that are not whole or do not
    // fill a group, follow one by one.  The order of the sum is that of the chunks either way.
    int c = c_lo;
    {
        const int whole = min(c_hi, K / FCH);
        int left = whole > c_lo ? (whole - c_lo) / U : 0;
        if (left > 0) {
            Rows x, y;
            load_group(c, x);
            while (left > 2) {
                load_group(c + U, y);
                group_products(x);
                load_group(c + 2 * U, x);
                group_products(y);
                c += 2 * U;
                left -= 2;
            }
            if (left == 2) {
                load_group(c + U, y);
                group_products(x);
                group_products(y);
                c += 2 * U;
            } else {
                group_products(x);
                c += U;
            }
        }
    }
    for (; c < c_hi; ++c) {
        f32x4 w[NT][2], a[MT][2];
        auto load_chunk = [&](auto four) {
#pragma unroll
            for (int h = 0; h < 2; ++h) {
#pragma unroll
                for (int nt = 0; nt < NT; ++nt) w[nt][h] = four(wrow[nt], c * FCH + 4 * h);
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) a[mt][h] = four(arow[mt], c * FCH + 4 * h);
            }
        };
        if ((c + 1) * FCH <= K)
            load_chunk([&](const float* p, int at) { return load4(p + at); });
        else if (K % 4 == 0)
            load_chunk([&](const float* p, int at) { return load_k4<PIECES>(p, at, 8 * g, K); });
        else
            load_chunk([&](const float* p, int at) { return load_k4<ELEMENTS>(p, at, 8 * g, K); });
        products(w, a);
    }

    // the runs are added in their order
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int i = 0; i < 4; ++i) red[wave][((nt * MT + mt) * 4 + i) * 64 + lane] = acc[nt][mt][i];
    __syncthreads();
    if constexpr (GLU) {
        for (int i = threadIdx.x; i < NT * MT * 128; i += FRUNS * RL_WAVE) {
            const int ln = i & 63, tile = i >> 7, j = (i >> 6) & 1, e = tile * 256 + j * 64 + ln;
            const int n = (n0 + tile / MT * 16) / 2 + 2 * (ln >> 4) + j;
            const int m = m0 + tile % MT * 16 + (ln & 15);
            if (n >= N || m >= M) continue;
            float v[2];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                v[h] = red[0][e + 128 * h];
#pragma unroll
                for (int w = 1; w < FRUNS; ++w) v[h] = w & 1 ? v[h] - red[w][e + 128 * h] : v[h] + red[w][e + 128 * h];
                v[h] = finite_or_wide(v[h], A + (size_t)m * lda, W + ((size_t)n + (h ? N : 0)) * ldw, K);
            }
            C[(size_t)m * ldc + n] = silu_mul(v[0], v[1]);
        }
        return;
    }
    for (int e = threadIdx.x; e < NT * MT * 256; e += FRUNS * RL_WAVE) {
        const int ln = e & 63, tile = e >> 8;
        const int n = n0 + tile / MT * 16 + 4 * (ln >> 4) + ((e >> 6) & 3);
        const int m = m0 + tile % MT * 16 + (ln & 15);
        if (n >= N || m >= M) continue;
        float v = red[0][e];
#pragma unroll
        for (int w = 1; w < FRUNS; ++w) v = w & 1 ? v - red[w][e] : v + red[w][e];
        C[(size_t)m * ldc + n] = finite_or_wide(v, A + (size_t)m * lda, W + (size_t)n * ldw, K);
    }
}

// The pairs of a wave's TN x TM blocks; row(y) and col(x): the lane's row, its first of two columns.  The few that are not
// finite stand behind, once.
template <int TN, int TM, typename ROW, typename COL>
__device__ __forceinline__ void gated_results(const f32x4 (&total)[TN][TM], float* C, const float* A, const float* W, int M, int N, int K,
                                              int lda, int ldw, int ldc, ROW row, COL col) {
    uint32_t wide = 0;
    static_assert(TN * TM * 2 <= 32, "a bit a pair");
    const bool pairs = (ldc & 1) == 0 && (reinterpret_cast<uintptr_t>(C) & 7) == 0;
#pragma unroll
    for (int x = 0; x < TN; ++x)
#pragma unroll
        for (int y = 0; y < TM; ++y) {
            const int m = row(y), n = col(x);
            if (m >= M) continue;
            f32x2 v;
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const float gate = total[x][y][j], up = total[x][y][2 + j];
                if (!__builtin_isfinite(gate) || !__builtin_isfinite(up)) wide |= 1u << ((x * TM + y) * 2 + j);
                v[j] = silu_mul(gate * DOWN, up * DOWN);
            }
            float* out = C + (size_t)m * ldc + n;
            if (pairs && n + 1 < N) {
                *reinterpret_cast<f32x2*>(out) = v;
            } else {
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    if (n + j < N) out[j] = v[j];
            }
        }
    while (wide) {
        const int e = __ffs(wide) - 1;
        wide &= wide - 1;
        float gate = 0.f, up = 0.f;
        int m = 0, n = 0;
#pragma unroll
        for (int x = 0; x < TN; ++x)
#pragma unroll
            for (int y = 0; y < TM; ++y)
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    if (e == (x * TM + y) * 2 + j) gate = total[x][y][j], up = total[x][y][2 + j], m = row(y), n = col(x) + j;
        if (n >= N) continue;
        const float* a = A + (size_t)m * lda;
        C[(size_t)m * ldc + n] = silu_mul(finite_or_wide(gate, a, W + (size_t)n * ldw, K), finite_or_wide(up, a, W + ((size_t)n + N) * ldw, K));
    }
}

// ---- more rows: tiles whose operands are split once and shared through LDS ---------------------
// A workgroup of four waves owns 32 TM x 32 TN results, a wave 16 TM x 16 TN of them.  A chunk's rows of
// A and W travel through registers, where they are split, into LDS in the order in which the matrix
// instruction's operands are read (16 rows x 8 k of a lane group are 16 bytes a lane, side by side), so
// that neither side meets a bank twice.  Large tiles: LDS holds one chunk, two workgroups a compute unit
// cover each other's barriers and the next chunk's rows are asked for before this one is multiplied.
// Small ones, whose chunks are short: LDS holds two chunks (one barrier a chunk), and three chunks' rows
// are on their way.
template <int TM, int TN, Length L, bool RUNS, bool GLU>
__global__ __launch_bounds__(256, 2) void gemm_f32_tile_kernel(
    const float* __restrict__ A, const float* __restrict__ W, float* __restrict__ C, int M, int N,
    int K, int lda, int ldw, int ldc, int tiles_m, int tiles_n, int runs) {
    constexpr int BM = 32 * TM, BN = 32 * TN;  // rows of A and of W a workgroup takes
    constexpr int PA = BM < 64 ? 1 : BM / 64, PW = BN / 64;  // pieces of 8 k that a thread carries
    constexpr int PLANE_A = BM * FCH, PLANE_W = BN * FCH;    // one operand's hi, mid or lo in LDS
    constexpr bool SMALL = TM * TN <= 4;
    constexpr int BUFS = SMALL ? 2 : 1, DEPTH = SMALL ? 3 : 1;
    __shared__ __align__(16) __bf16 lds_a[BUFS][3 * PLANE_A], lds_w[BUFS][3 * PLANE_W];

    const int lane = threadIdx.x & (RL_WAVE - 1);
    const int wave = threadIdx.x / RL_WAVE;
    const int r16 = lane & 15;
    const int g = lane >> 4;

    // Tiles in groups of eight row blocks, row blocks fastest; a die (workgroups i, i + 8, ..) takes
    // a contiguous share of them, so that the tiles it works on at a time share their operands in its L2.
    const int tiles = tiles_m * tiles_n;
    int t = blockIdx.x;
    {
        const int share = tiles / 8, rest = tiles % 8, die = t % 8;
        t = die * share + min(die, rest) + t / 8;
    }
    const int band = t / (8 * tiles_n), first = band * 8, high = min(8, tiles_m - first);
    const int m0 = (first + t % (8 * tiles_n) % high) * BM;
    const int n0 = t % (8 * tiles_n) / high * BN;

    const int piece = threadIdx.x & 3;  // the lane group a thread's pieces belong to
    const float *from_a[PA], *from_w[PW];
    int to_a[PA], to_w[PW];
    auto place = [&](int row) { return (row >> 4) * 512 + (piece * 16 + ((row & 15) ^ (2 * piece))) * 8; };
#pragma unroll
    for (int i = 0; i < PA; ++i) {
        const int row = ((threadIdx.x >> 2) & (BM - 1)) + 64 * i;  // 32 rows: two threads carry the same piece
        from_a[i] = A + (size_t)min(m0 + row, M - 1) * lda + 8 * piece;
        to_a[i] = place(row);
    }
#pragma unroll
    for (int i = 0; i < PW; ++i) {
        const int row = (threadIdx.x >> 2) + 64 * i;
        from_w[i] = W + row_of<GLU>(n0 + row, N) * ldw + 8 * piece;
        to_w[i] = place(row);
    }
    const int wm = (wave & 1) * TM, wn = (wave >> 1) * TN;  // the wave's first 16-row blocks
    const int at = (g * 16 + (r16 ^ (2 * g))) * 8;

    const int chunks = (K + FCH - 1) / FCH;
    const int per = (chunks + FRUNS - 1) / FRUNS;
    const int run_lo = RUNS ? blockIdx.y * runs : 0, run_hi = RUNS ? run_lo + runs : FRUNS;
    const int begin = min(chunks, run_lo * per), end = min(chunks, run_hi * per);
    int run = run_lo;
    int next = begin, stored = run_lo;  // the chunk that goes to LDS next, and its run

    struct Raw {
        f32x4 a[PA][2], w[PW][2];
    };
    auto load = [&](int c, Raw& r) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
#pragma unroll
            for (int i = 0; i < PA; ++i) r.a[i][h] = load_k4<L>(from_a[i], c * FCH + 4 * h, 8 * piece, K);
#pragma unroll
            for (int i = 0; i < PW; ++i) r.w[i][h] = load_k4<L>(from_w[i], c * FCH + 4 * h, 8 * piece, K);
        }
    };
    auto store = [&](const Raw& r, int buf) {
        const float up = stored & 1 ? -UP : UP;
        if (++next == (stored + 1) * per) ++stored;
#pragma unroll
        for (int i = 0; i < PA; ++i) {
            const Split s = split8(r.a[i][0], r.a[i][1], up);
#pragma unroll
            for (int p = 0; p < 3; ++p) *reinterpret_cast<bf16x8*>(&lds_a[buf][p * PLANE_A + to_a[i]]) = s.p[p];
        }
#pragma unroll
        for (int i = 0; i < PW; ++i) {
            const Split s = split8(r.w[i][0], r.w[i][1]);
#pragma unroll
            for (int p = 0; p < 3; ++p) *reinterpret_cast<bf16x8*>(&lds_w[buf][p * PLANE_W + to_w[i]]) = s.p[p];
        }
    };
    f32x4 acc[TN][TM], total[TN][TM];
    auto products = [&](int buf) {
        bf16x8 w[TN][3];
#pragma unroll
        for (int x = 0; x < TN; ++x)
#pragma unroll
            for (int p = 0; p < 3; ++p)
                w[x][p] = *reinterpret_cast<const bf16x8*>(&lds_w[buf][p * PLANE_W + (wn + x) * 512 + at]);
        // neighbouring instructions belong to different sums: YB TN of them stand between two of one
        constexpr int YB = SMALL ? TM : 1;
#pragma unroll
        for (int y0 = 0; y0 < TM; y0 += YB) {
            bf16x8 a[YB][3];
#pragma unroll
            for (int y = 0; y < YB; ++y)
#pragma unroll
                for (int p = 0; p < 3; ++p)
                    a[y][p] = *reinterpret_cast<const bf16x8*>(&lds_a[buf][p * PLANE_A + (wm + y0 + y) * 512 + at]);
#pragma unroll
            for (int s = 0; s < 6; ++s)
#pragma unroll
                for (int y = 0; y < YB; ++y)
#pragma unroll
                    for (int x = 0; x < TN; ++x)
                        acc[x][y0 + y] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                            w[x][PIECE_W[s]], a[y][PIECE_A[s]], acc[x][y0 + y], 0, 0, 0);
        }
    };

    auto zero = [&]() {
#pragma unroll
        for (int x = 0; x < TN; ++x)
#pragma unroll
            for (int y = 0; y < TM; ++y) acc[x][y] = (f32x4){0.f, 0.f, 0.f, 0.f};
    };
    // the run is over: its result joins the total, or goes as it is to the kernel that adds the runs
    auto finish_run = [&]() {
#pragma unroll
        for (int x = 0; x < TN; ++x)
#pragma unroll
            for (int y = 0; y < TM; ++y) {
                if (!RUNS) {
                    total[x][y] = run == 0 ? acc[x][y] : run & 1 ? total[x][y] - acc[x][y] : total[x][y] + acc[x][y];
                    continue;
                }
                const int m = m0 + (wm + y) * 16 + r16, n = n0 + (wn + x) * 16 + 4 * g;
                if (m >= M) continue;
                float* out = C + ((size_t)run * M + m) * N + n;
                if ((N & 3) == 0 && n < N) {
                    *reinterpret_cast<f32x4*>(out) = acc[x][y];
                } else {
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        if (n + i < N) out[i] = acc[x][y][i];
                }
            }
        ++run;
        zero();
    };
    zero();
    if (begin < end) {
        Raw raw[DEPTH];
        if (SMALL) {
            load(begin, raw[0]);
            store(raw[0], 0);
#pragma unroll
            for (int d = 0; d < DEPTH; ++d) load(min(begin + 1 + d, end - 1), raw[d]);
            __syncthreads();
            int left = end - begin, c = begin, buf = 0;
            auto step = [&](Raw& r) {
                store(r, buf ^ 1);  // chunk c + 1 (the last chunk once more at the end: nobody reads it)
                load(min(c + 1 + DEPTH, end - 1), r);
                products(buf);
                ++c;
                buf ^= 1;
                if (c == (run + 1) * per || c == end) finish_run();
                __syncthreads();
            };
            while (left >= DEPTH) {
#pragma unroll
                for (int d = 0; d < DEPTH; ++d) step(raw[d]);
                left -= DEPTH;
            }
#pragma unroll
            for (int d = 0; d < DEPTH - 1; ++d)
                if (d < left) step(raw[d]);
        } else {
            load(begin, raw[0]);
            for (int c = begin; c < end;) {
                store(raw[0], 0);
                __syncthreads();
                load(min(c + 1, end - 1), raw[0]);
                products(0);
                ++c;
                if (c == (run + 1) * per || c == end) finish_run();
                __syncthreads();
            }
        }
    }
    while (run < run_hi) finish_run();  // runs without a chunk: zeros
    if (RUNS) return;
    if constexpr (GLU) {
        gated_results<TN, TM>(total, C, A, W, M, N, K, lda, ldw, ldc, [&](int y) { return m0 + (wm + y) * 16 + r16; },
                              [&](int x) { return (n0 + (wn + x) * 16) / 2 + 2 * g; });
        return;
    }
    // which of the lane's results are not finite: they are few or none, so their sums stand behind, once
    uint64_t wide = 0;
    const bool pieces = (ldc & 3) == 0 && (reinterpret_cast<uintptr_t>(C) & 15) == 0;
#pragma unroll
    for (int x = 0; x < TN; ++x)
#pragma unroll
        for (int y = 0; y < TM; ++y) {
            const int m = m0 + (wm + y) * 16 + r16, n = n0 + (wn + x) * 16 + 4 * g;
            if (m >= M) continue;
            f32x4 v;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if (!__builtin_isfinite(total[x][y][i])) wide |= 1ull << ((x * TM + y) * 4 + i);
                v[i] = total[x][y][i] * DOWN;
            }
            float* out = C + (size_t)m * ldc + n;
            if (pieces && n + 3 < N) {
                *reinterpret_cast<f32x4*>(out) = v;
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (n + i < N) out[i] = v[i];
            }
        }
    while (wide) {
        const int e = __ffsll((unsigned long long)wide) - 1;
        wide &= wide - 1;
        const int m = m0 + (wm + (e >> 2) % TM) * 16 + r16, n = n0 + (wn + (e >> 2) / TM) * 16 + 4 * g + (e & 3);
        if (n < N) C[(size_t)m * ldc + n] = wide_sum(A + (size_t)m * lda, W + (size_t)n * ldw, K);
    }
}

// ---- some rows: a wave a run, nothing shared ------------------------------------------
// The tiles above walk K as a chain of chunks, each split, stored to LDS, waited for and read back, or leave their runs to
// a second kernel.  Here the eight waves of a workgroup hold the same 16 NT x 16 MT results, each over its run of K, and no
// wave waits for another.  A wave's rows go from memory straight into its own part of LDS, eight lanes a row (asked for into
// registers as the instruction takes them, lane by lane from another row, a unit gets 16 bytes a cycle: 6,144 x 4,096 at 225 rows
// 87 us, so 77), and from there to its registers, where they are split; a place is asked for again as soon as it has been
// read, one chunk ahead or two.
// What bounds it: splitting and multiplying, 208 (NT + MT) and 96 NT MT cycles a wave and chunk, which take about as long as
// one after the other (at 225 rows of 6,144 x 4,096 the splits alone 38 us, the loads alone 43, all 77), so the tiles
// are as large as the rows and the number of units allow.  The next split between the products 77 -> 74, the first four waves
// ahead of the others on their SIMDs 60 -> 56 (4,096 x 4,096).
// Microseconds, the other kernels / this: ops.f32_waves; steps, together with the gated products' own activation: 0.6B three
// prompts of 225 tokens 3,613 / 2,804, 8B eight requests decode 7,465 / 6,903.
typedef __attribute__((address_space(3))) void* rl_lds_ptr;
#define RUNS_LDS (160 * 1024)

// Sixteen rows' chunks from LDS, the lane's eight k each; the wait stands in the block that asks, so that the compiler adds
// none for loads that are on their way into LDS.
__device__ __forceinline__ void read_rows(f32x4 (&r)[1][2], uint32_t at) {
    asm volatile("ds_read_b128 %0, %2\n ds_read_b128 %1, %3\n s_waitcnt lgkmcnt(0)" : "=&v"(r[0][0]), "=&v"(r[0][1]) : "v"(at), "v"(at ^ 16) : "memory");
}
__device__ __forceinline__ void read_rows(f32x4 (&r)[2][2], uint32_t at) {
    asm volatile(
        "ds_read_b128 %0, %4\n ds_read_b128 %1, %5\n ds_read_b128 %2, %4 offset:2048\n ds_read_b128 %3, %5 offset:2048\n s_waitcnt lgkmcnt(0)"
        : "=&v"(r[0][0]), "=&v"(r[0][1]), "=&v"(r[1][0]), "=&v"(r[1][1])
        : "v"(at), "v"(at ^ 16)
        : "memory");
}

template <int NT, int MT, bool GLU>
__global__ __launch_bounds__(FRUNS* RL_WAVE) void gemm_f32_runs_kernel(
    const float* __restrict__ A, const float* __restrict__ W, float* __restrict__ C, int M, int N, int K, int lda, int ldw,
    int ldc, int tiles_m, int tiles_n) {
#if defined(__HIP_DEVICE_COMPILE__)  // (the host pass does not know the LDS loads)
    constexpr int T = NT + MT, SLOT = 2048, CHUNK = T * SLOT;  // a place: sixteen rows' chunk
    // One chunk ahead, so that a unit holds two workgroups of tiles of up to eight blocks and five places, 64 to 80 KB each ((4, 2)
    // and (6, 1) take 96 and 112 KB, more blocks 128 and more for the sums alone); two for the smallest tile, whose chunk does not
    // cover memory's answer.  (Three as far as they fit / this, us: 8 rows of 4,096 x 12,288 43.0 / 39.5, 6,144 x 4,096 22.9 / 21.4; 225 of
    // 1,024 x 3,072 19.5 / 17.9, of 1,536 x 512 10.8 / 7.9; one for the smallest too: 8 rows of 4,096 x 4,096 14.8 / 16.3; two at (1, 2), 96 KB: 17 / 32 rows
    // of 4,096 x 1,024 7.0 / 6.4, 8.3 / 7.7, of 4,096 x 4,096 20.1 / 19.5, 22.5 / 21.4.)
    constexpr int D = NT == 1 && MT == 1 ? 2 : 1;
    constexpr int GA = MT % 2 ? 1 : 2, GW = NT % 2 ? 1 : 2;  // places read together
    constexpr int BLOCKS = NT * MT, ROUNDS = (BLOCKS + FRUNS - 1) / FRUNS;
    static_assert(FRUNS * D * CHUNK <= RUNS_LDS && 2 * D * T <= 64, "the chunks fit, and the counter");
    constexpr int SUMS = (ROUNDS > 1 ? 2 : 1) * FRUNS * FRUNS * RL_WAVE * 16, BYTES = FRUNS * D * CHUNK > SUMS ? FRUNS * D * CHUNK : SUMS;
    static_assert(BLOCKS > FRUNS || T > 5 || 2 * BYTES <= RUNS_LDS, "two workgroups a unit");
    __shared__ __attribute__((aligned(1024))) unsigned char lds[BYTES];

    const int lane = threadIdx.x & (RL_WAVE - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / RL_WAVE);
    const int r16 = lane & 15, g = lane >> 4;
    // the order of the tiles: as in gemm_f32_tile_kernel
    const int tiles = tiles_m * tiles_n;
    int t = blockIdx.x;
    {
        const int share = tiles / 8, rest = tiles % 8, die = t % 8;
        t = die * share + min(die, rest) + t / 8;
    }
    const int band = t / (8 * tiles_n), first = band * 8, high = min(8, tiles_m - first);
    const int m0 = (first + t % (8 * tiles_n) % high) * (16 * MT);
    const int n0 = t % (8 * tiles_n) / high * (16 * NT);

    const int chunks = K / FCH, per = (chunks + FRUNS - 1) / FRUNS;
    const int c_lo = min(chunks, wave * per), c_hi = min(chunks, c_lo + per);

    // A load lays a wave's 64 x 16 bytes side by side: eight rows, unit u of row r at u ^ (r / 2), so that reads meet every
    // bank once.  Rows beyond the matrices find no records: zeros, whose results are dropped.
    const int row0 = GLU ? n0 / 2 : n0;
    const uint32_t w_bytes = ((uint32_t)((GLU ? 2 * N : N) - row0 - 1) * ldw + K) * 4, a_bytes = ((uint32_t)(M - m0 - 1) * lda + K) * 4;
    const float *w_from = W + (size_t)row0 * ldw, *a_from = A + (size_t)m0 * lda;
    uint32_t w_off[2], a_off[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int r = 8 * i + (lane >> 3);
        const uint32_t unit = ((lane & 7) ^ (r >> 1)) * 16;
        w_off[i] = (uint32_t)(GLU ? ((r >> 1) & 6) + (r & 1) + (r & 2 ? N : 0) : r) * (uint32_t)ldw * 4 + unit;
        a_off[i] = (uint32_t)r * (uint32_t)lda * 4 + unit;
    }
    const uint32_t w_step = (uint32_t)(GLU ? 8 : 16) * (uint32_t)ldw * 4, a_step = 16 * (uint32_t)lda * 4;
    unsigned char* const own = lds + wave * (D * CHUNK);
    // the rows of places MT .. MT + NT - 1 are W's; behind the last chunk no records are found, and no chunk is asked for: the
    // unit compares a load's own offset with the records less the scalar offset, which would wrap
    auto ask = [&](int place, int c, uint32_t at) {
        const bool is_a = place < MT, there = c < c_hi;
        const auto rs = is_a ? __builtin_amdgcn_make_buffer_rsrc((void*)a_from, 0, there ? a_bytes : 0u, 0x00020000)
                             : __builtin_amdgcn_make_buffer_rsrc((void*)w_from, 0, there ? w_bytes : 0u, 0x00020000);
        const int chunk = there ? c * (FCH * 4) : 0;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const uint32_t off = is_a ? a_off[i] + place * a_step : w_off[i] + (place - MT) * w_step;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (rl_lds_ptr)(own + at + place * SLOT + i * 1024), 16, off, chunk, 0, 0);
        }
    };

    f32x4 acc[NT][MT];
#pragma unroll
    for (int x = 0; x < NT; ++x)
#pragma unroll
        for (int y = 0; y < MT; ++y) acc[x][y] = (f32x4){0.f, 0.f, 0.f, 0.f};

#pragma unroll
    for (int d = 0; d < D; ++d)
#pragma unroll
        for (int p = 0; p < T; ++p) ask(p, c_lo + d, d * CHUNK);
    const uint32_t l0 = (uint32_t)(uintptr_t)(rl_lds_ptr)own + r16 * 128 + ((2 * g) ^ (r16 >> 1)) * 16;
    const float up = wave & 1 ? -UP : UP;
    uint32_t at = 0;
    if (wave < 4) __builtin_amdgcn_s_setprio(1);  // a SIMD's two waves split and multiply in turn rather than both at a time
#pragma unroll 1
    for (int c = c_lo; c < c_hi; ++c) {
        // of the newest 2 D T loads all but those of the places read next may be missing
        Split as[MT];
#pragma unroll
        for (int y = 0; y < MT; y += GA) {
            f32x4 raw[GA][2];
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * (D * T - GA)) : "memory");
            read_rows(raw, l0 + at + y * SLOT);
#pragma unroll
            for (int j = 0; j < GA; ++j) ask(y + j, c + D, at);
#pragma unroll
            for (int j = 0; j < GA; ++j) as[y + j] = split8(raw[j][0], raw[j][1], up);
        }
        Split ws[2][GW];
        auto take = [&](int x, Split (&to)[GW]) {
            f32x4 raw[GW][2];
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * (D * T - GW)) : "memory");
            read_rows(raw, l0 + at + (MT + x) * SLOT);
#pragma unroll
            for (int j = 0; j < GW; ++j) ask(MT + x + j, c + D, at);
#pragma unroll
            for (int j = 0; j < GW; ++j) to[j] = split8(raw[j][0], raw[j][1]);
        };
        take(0, ws[0]);
#pragma unroll
        for (int x = 0; x < NT; x += GW) {
            __builtin_amdgcn_sched_barrier(0);
            if (x + GW < NT) take(x + GW, ws[(x / GW + 1) & 1]);
#pragma unroll
            for (int s = 0; s < 6; ++s)
#pragma unroll
                for (int j = 0; j < GW; ++j)
#pragma unroll
                    for (int y = 0; y < MT; ++y)
                        acc[x + j][y] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ws[x / GW & 1][j].p[PIECE_W[s]], as[y].p[PIECE_A[s]], acc[x + j][y], 0, 0, 0);
            if (x + GW < NT) {  // three vector instructions of the next split behind every product
#pragma unroll
                for (int i = 0; i < 6 * GW * MT; ++i) {
                    __builtin_amdgcn_sched_group_barrier(8, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(2, 3, 0);
                }
            }
        }
        at = at == (D - 1) * CHUNK ? 0 : at + CHUNK;
    }
    __builtin_amdgcn_s_setprio(0);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // nothing may still be on its way to where the sums go
    __syncthreads();

    // The runs are added in their order, a block a wave, eight blocks a round.
    f32x4* const sums = reinterpret_cast<f32x4*>(lds);  // [2][block][run][lane]
#pragma unroll
    for (int round = 0; round < ROUNDS; ++round) {
        f32x4* const here = sums + (round & 1) * (FRUNS * FRUNS * RL_WAVE) + lane;
#pragma unroll
        for (int b = 0; b < FRUNS; ++b)
            if (FRUNS * round + b < BLOCKS) here[(b * FRUNS + wave) * RL_WAVE] = acc[(FRUNS * round + b) / MT][(FRUNS * round + b) % MT];
        __syncthreads();
        const int block = FRUNS * round + wave;
        if (block >= BLOCKS) break;
        f32x4 total[1][1];
        total[0][0] = here[wave * FRUNS * RL_WAVE];
#pragma unroll
        for (int r = 1; r < FRUNS; ++r) {
            const f32x4 v = here[(wave * FRUNS + r) * RL_WAVE];
            total[0][0] = r & 1 ? total[0][0] - v : total[0][0] + v;
        }
        const int m = m0 + block % MT * 16 + r16, n = n0 + block / MT * 16 + (GLU ? 0 : 4 * g);
        if constexpr (GLU) {
            gated_results<1, 1>(total, C, A, W, M, N, K, lda, ldw, ldc, [&](int) { return m; }, [&](int) { return n / 2 + 2 * g; });
        } else if (m < M) {
            f32x4 v;
#pragma unroll
            for (int i = 0; i < 4; ++i) v[i] = n + i < N ? finite_or_wide(total[0][0][i], A + (size_t)m * lda, W + (size_t)(n + i) * ldw, K) : 0.f;
            float* out = C + (size_t)m * ldc + n;
            if ((ldc & 3) == 0 && (reinterpret_cast<uintptr_t>(C) & 15) == 0 && n + 3 < N) {
                *reinterpret_cast<f32x4*>(out) = v;
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (n + i < N) out[i] = v[i];
            }
        }
    }
#endif
}

// ---- many rows: the pieces of A laid out before, eight waves in two halves ----------------------
// One kernel splits A once, instead of every workgroup that reads its rows, and lays the pieces down as the matrix
// instruction reads them (bound by memory, 10 bytes an element: 10 us for 2,048 x 4,096): [16 rows][chunk][hi, mid, lo][64 lanes][8 k], 1 KB a piece.  Rows behind the last are zeros.
__global__ __launch_bounds__(256) void gemm_f32_pieces_kernel(const float* __restrict__ A, __bf16* __restrict__ P, int M,
                                                              int chunks, int lda, int per) {
    const int lane = threadIdx.x & (RL_WAVE - 1), r16 = lane & 15, g = lane >> 4;
    const int block = blockIdx.y, c = blockIdx.x * 4 + threadIdx.x / RL_WAVE;
    if (c >= chunks) return;
    const int row = block * 16 + r16;
    f32x4 x = {0.f, 0.f, 0.f, 0.f}, y = x;
    if (row < M) {
        const float* p = A + (size_t)row * lda + c * FCH + 8 * g;
        x = load4(p), y = load4(p + 4);
    }
    const Split s = split8(x, y, c / per & 1 ? -UP : UP);
    __bf16* out = P + ((size_t)block * chunks + c) * 1536 + lane * 8;
#pragma unroll
    for (int p = 0; p < 3; ++p) *reinterpret_cast<bf16x8*>(out + p * 512) = s.p[p];
}

#define WIDE_A (256 * FCH * 6)  // bytes of a chunk's pieces of A

template <int N>
__device__ __forceinline__ void wait_loads() {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
__device__ __forceinline__ void turn() {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
}
// operand reads wait in the block that asks, so that the compiler adds no wait for loads that are on their way into LDS
__device__ __forceinline__ void read_w(bf16x8 (&w)[4][3], uint32_t at) {
    asm volatile(
        "ds_read_b128 %0, %12\n ds_read_b128 %1, %12 offset:8192\n ds_read_b128 %2, %12 offset:16384\n"
        "ds_read_b128 %3, %12 offset:1024\n ds_read_b128 %4, %12 offset:9216\n ds_read_b128 %5, %12 offset:17408\n"
        "ds_read_b128 %6, %12 offset:2048\n ds_read_b128 %7, %12 offset:10240\n ds_read_b128 %8, %12 offset:18432\n"
        "ds_read_b128 %9, %12 offset:3072\n ds_read_b128 %10, %12 offset:11264\n ds_read_b128 %11, %12 offset:19456\n"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(w[0][0]), "=&v"(w[0][1]), "=&v"(w[0][2]), "=&v"(w[1][0]), "=&v"(w[1][1]), "=&v"(w[1][2]),
          "=&v"(w[2][0]), "=&v"(w[2][1]), "=&v"(w[2][2]), "=&v"(w[3][0]), "=&v"(w[3][1]), "=&v"(w[3][2])
        : "v"(at)
        : "memory");
}
__device__ __forceinline__ void read_w(bf16x8 (&w)[3][3], uint32_t at) {
    asm volatile(
        "ds_read_b128 %0, %9\n ds_read_b128 %1, %9 offset:6144\n ds_read_b128 %2, %9 offset:12288\n"
        "ds_read_b128 %3, %9 offset:1024\n ds_read_b128 %4, %9 offset:7168\n ds_read_b128 %5, %9 offset:13312\n"
        "ds_read_b128 %6, %9 offset:2048\n ds_read_b128 %7, %9 offset:8192\n ds_read_b128 %8, %9 offset:14336\n"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(w[0][0]), "=&v"(w[0][1]), "=&v"(w[0][2]), "=&v"(w[1][0]), "=&v"(w[1][1]), "=&v"(w[1][2]),
          "=&v"(w[2][0]), "=&v"(w[2][1]), "=&v"(w[2][2])
        : "v"(at)
        : "memory");
}
__device__ __forceinline__ void read_a2(bf16x8 (&a)[2][3], uint32_t at) {
    asm volatile(
        "ds_read_b128 %0, %6\n ds_read_b128 %1, %6 offset:1024\n ds_read_b128 %2, %6 offset:2048\n"
        "ds_read_b128 %3, %6 offset:3072\n ds_read_b128 %4, %6 offset:4096\n ds_read_b128 %5, %6 offset:5120\n"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(a[0][0]), "=&v"(a[0][1]), "=&v"(a[0][2]), "=&v"(a[1][0]), "=&v"(a[1][1]), "=&v"(a[1][2])
        : "v"(at)
        : "memory");
}

// The tiles above with 256 rows of A and 32 TN of W a workgroup, 64 x 16 TN a wave; the same sums in the same order.  What
// bounds it: the matrix cores at the clock they hold with real operands (2,048 rows of 24,576 x 4,096 run at 1.51
// PFLOP/s of bfloat16, a large bfloat16 product at 1.54), so everything else is kept out of their way:
//   * A's pieces go from memory straight into LDS, no wave splits a row of A; W, whose pieces would be half as many bytes
//     again as it, is split by the workgroup, 8 k of a row a thread: 60 vector instructions a chunk beside 96 products.
//   * The waves are two halves that take turns: while one multiplies (48 products), the other reads its next operands,
//     splits and stores W's next chunk and asks memory for later ones.  A barrier ends each turn, the second half begins
//     one barrier later.
//   * A chunk is two turns, each with half of the wave's rows of A, so every half has a place of its own in LDS and is
//     asked for one and a half chunks ahead; W one chunk ahead, through registers.  Nothing waits for all loads.
//   * No bank is met twice: A lies as it is read, W's rows are permuted as in the kernel above.
// Microseconds at 2,048 rows, the tiles of 128 x 128 / this with A's pieces made: 6,144 x 4,096 521 / 453, 4,096 x 4,096
// 326 / 279, 24,576 x 4,096 1,957 / 1,624, 4,096 x 12,288 1,006 / 817.  TN = 3 is for matrices whose tiles of
// 128 columns leave a short last round (ops.f32_wide has the rule).
template <int TN, bool GLU>
__global__ __launch_bounds__(512) void gemm_f32_wide_kernel(const float* __restrict__ A, const __bf16* __restrict__ P,
                                                            const float* __restrict__ W, float* __restrict__ C, int M,
                                                            int N, int K, int lda, int ldw, int ldc, int tiles_m,
                                                            int tiles_n) {
#if defined(__HIP_DEVICE_COMPILE__)  // (the host pass does not know the LDS loads)
    constexpr int BN = 32 * TN, PLANE_W = BN * FCH * 2, WIDE_W = 3 * PLANE_W;
    // [2][16 blocks][3 pieces][1 KB] of A, [2][3 pieces][2 TN blocks][1 KB] of W
    __shared__ __attribute__((aligned(1024))) unsigned char lds[2 * WIDE_A + 2 * WIDE_W];
    const int tid = threadIdx.x, lane = tid & (RL_WAVE - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid / RL_WAVE);
    const int r16 = lane & 15, g = lane >> 4;
    const int wm = wave >> 1, wn = wave & 1;  // the wave's rows of A, of W

    // the order of the tiles: as in gemm_f32_tile_kernel
    const int tiles = tiles_m * tiles_n;
    int t = blockIdx.x;
    {
        const int share = tiles / 8, rest = tiles % 8, die = t % 8;
        t = die * share + min(die, rest) + t / 8;
    }
    const int band = t / (8 * tiles_n), first = band * 8, high = min(8, tiles_m - first);
    const int tm = first + t % (8 * tiles_n) % high, m0 = tm * 256;
    const int n0 = t % (8 * tiles_n) / high * BN;

    const int chunks = K / FCH, per = (chunks + FRUNS - 1) / FRUNS;

    // A: 48 pieces a chunk, three loads a wave and turn: blocks 2 j and 2 j + 1 of every wave's four (j: turn)
    const int blocks = min(16, (M + 15) / 16 - tm * 16);  // that exist
    const uint32_t block_bytes = (uint32_t)chunks * 3072;
    auto rs_a = __builtin_amdgcn_make_buffer_rsrc((void*)((const char*)P + (size_t)tm * 16 * block_bytes), 0, blocks * block_bytes, 0x00020000);
    uint32_t a_from[3], a_to[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        const int j = wave * 3 + i, block = j / 6 * 4 + j % 6 / 3, piece = j % 3;  // of turn 0; turn 1: two blocks on
        a_from[i] = block * block_bytes + piece * 1024 + lane * 16;
        a_to[i] = block * 3072 + piece * 1024;
    }
    auto load_a = [&](int c, int j) {  // (behind the last chunk: that again, nobody reads it)
        const uint32_t off = (uint32_t)min(c, chunks - 1) * 3072 + 2 * j * block_bytes;
#pragma unroll
        for (int i = 0; i < 3; ++i)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rs_a, (rl_lds_ptr)(lds + (c & 1) * WIDE_A + a_to[i] + 2 * j * 3072), 16, a_from[i] + off, 0, 0, 0);
    };
    // W: 8 k of a row a thread, through registers (where the rows are fewer, the last threads carry what others do:
    // every wave has the same loads on their way)
    const int piece = tid & 3, row = (tid >> 2) < BN ? tid >> 2 : (tid >> 2) - 32;
    const float* from_w = W + row_of<GLU>(n0 + row, N) * ldw + 8 * piece;
    unsigned char* to_w = lds + 2 * WIDE_A + (row >> 4) * 1024 + (piece * 16 + ((row & 15) ^ (2 * piece))) * 16;
    f32x4 raw[2];
    auto load_w = [&](int c) {
        const float* p = from_w + min(c, chunks - 1) * FCH;
        raw[0] = load4(p), raw[1] = load4(p + 4);
    };
    auto store_w = [&](int c) {
        const Split s = split8(raw[0], raw[1]);
#pragma unroll
        for (int p = 0; p < 3; ++p) {
            const uint32_t at = (uint32_t)(uintptr_t)(rl_lds_ptr)(to_w + (c & 1) * WIDE_W);
            asm volatile("ds_write_b128 %0, %1 offset:%2" ::"v"(at), "v"(s.p[p]), "n"(p * PLANE_W) : "memory");
        }
    };

    const uint32_t l0 = (uint32_t)(uintptr_t)(rl_lds_ptr)lds;
    const uint32_t w_at = l0 + 2 * WIDE_A + wn * TN * 1024 + (g * 16 + (r16 ^ (2 * g))) * 16;
    const uint32_t a_at = l0 + wm * 4 * 3072 + lane * 16;

    f32x4 acc[TN][4], total[TN][4];
    bf16x8 w[TN][3], a[2][3];
    auto products = [&](auto y0c) {
        constexpr int y0 = decltype(y0c)::value;
        turn();
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int s = 0; s < 6; ++s)
#pragma unroll
            for (int y = 0; y < 2; ++y)
#pragma unroll
                for (int x = 0; x < TN; ++x)
                    acc[x][y0 + y] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[x][PIECE_W[s]], a[y][PIECE_A[s]], acc[x][y0 + y], 0, 0, 0);
        __builtin_amdgcn_s_setprio(0);
        turn();
    };
#pragma unroll
    for (int x = 0; x < TN; ++x)
#pragma unroll
        for (int y = 0; y < 4; ++y) acc[x][y] = total[x][y] = (f32x4){0.f, 0.f, 0.f, 0.f};

    load_w(0);
    load_a(0, 0);
    load_a(0, 1);
    store_w(0);
    load_w(1);
    load_a(1, 0);
    wait_loads<5>();
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    turn();
    if (wave >= 4) __builtin_amdgcn_s_barrier();  // the second half is one turn behind
    __builtin_amdgcn_sched_barrier(0);

    int run = 0, left = per;  // chunks until the run is over
    auto finish_run = [&]() {
        const float sign = run & 1 ? -1.f : 1.f;
#pragma unroll
        for (int x = 0; x < TN; ++x)
#pragma unroll
            for (int y = 0; y < 4; ++y) {
#pragma unroll
                for (int i = 0; i < 4; ++i) total[x][y][i] = fmaf(acc[x][y][i], sign, total[x][y][i]);
                acc[x][y] = (f32x4){0.f, 0.f, 0.f, 0.f};
            }
        ++run;
        left = per;
    };
#pragma unroll 1
    for (int c = 0; c < chunks; ++c) {
        // all of W, half of A; the other half's place for the next chunk has been read
        load_a(c + 1, 1);
        read_w(w, w_at + (c & 1) * WIDE_W);
        read_a2(a, a_at + (c & 1) * WIDE_A);
        wait_loads<8>();  // this chunk's second half of A is there
        products(std::integral_constant<int, 0>{});
        // the other half of A; W's next chunk goes to LDS
        read_a2(a, a_at + (c & 1) * WIDE_A + 2 * 3072);
        store_w(c + 1);
        load_w(c + 2);
        load_a(c + 2, 0);
        wait_loads<8>();  // the next chunk's first half of A
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        products(std::integral_constant<int, 2>{});
        if (--left == 0 || c + 1 == chunks) finish_run();
    }
    while (run < FRUNS) finish_run();  // runs without a chunk: zeros
    wait_loads<0>();  // nothing may still be on its way into LDS when it is given back
    if (wave < 4) __builtin_amdgcn_s_barrier();

    if constexpr (GLU) {
        gated_results<TN, 4>(total, C, A, W, M, N, K, lda, ldw, ldc, [&](int y) { return m0 + wm * 64 + y * 16 + r16; },
                             [&](int x) { return (n0 + (wn * TN + x) * 16) / 2 + 2 * g; });
        return;
    }
    uint64_t wide = 0;
    const bool whole = (ldc & 3) == 0 && (reinterpret_cast<uintptr_t>(C) & 15) == 0;
#pragma unroll
    for (int x = 0; x < TN; ++x)
#pragma unroll
        for (int y = 0; y < 4; ++y) {
            const int m = m0 + wm * 64 + y * 16 + r16, n = n0 + (wn * TN + x) * 16 + 4 * g;
            if (m >= M) continue;
            f32x4 v;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if (!__builtin_isfinite(total[x][y][i])) wide |= 1ull << ((x * 4 + y) * 4 + i);
                v[i] = total[x][y][i] * DOWN;
            }
            float* out = C + (size_t)m * ldc + n;
            if (whole && n + 3 < N) {
                *reinterpret_cast<f32x4*>(out) = v;
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (n + i < N) out[i] = v[i];
            }
        }
    while (wide) {
        const int e = __ffsll((unsigned long long)wide) - 1;
        wide &= wide - 1;
        const int m = m0 + wm * 64 + (e >> 2) % 4 * 16 + r16, n = n0 + (wn * TN + (e >> 4)) * 16 + 4 * g + (e & 3);
        if (n < N) C[(size_t)m * ldc + n] = wide_sum(A + (size_t)m * lda, W + (size_t)n * ldw, K);
    }
#endif
}

// the runs of the tile kernel added in their order
template <bool GLU>
__global__ __launch_bounds__(256) void gemm_f32_add_runs_kernel(
    const float* __restrict__ parts, const float* __restrict__ A, const float* __restrict__ W,
    float* __restrict__ C, int M, int N, int K, int lda, int ldw, int ldc) {
    const int m = blockIdx.y;
    const int n = blockIdx.x * 256 + threadIdx.x;
    if (n >= (GLU ? N / 2 : N)) return;  // (a gated product's parts hold the gate's and up's columns)
    float run[GLU ? 2 : 1][FRUNS], v[GLU ? 2 : 1];
#pragma unroll
    for (int h = 0; h < (GLU ? 2 : 1); ++h)
#pragma unroll
        for (int r = 0; r < FRUNS; ++r) run[h][r] = parts[((size_t)r * M + m) * N + n + h * (N / 2)];
#pragma unroll
    for (int h = 0; h < (GLU ? 2 : 1); ++h) {
        v[h] = run[h][0];
#pragma unroll
        for (int r = 1; r < FRUNS; ++r) v[h] = r & 1 ? v[h] - run[h][r] : v[h] + run[h][r];
        v[h] = finite_or_wide(v[h], A + (size_t)m * lda, W + ((size_t)n + h * (N / 2)) * ldw, K);
    }
    if constexpr (GLU)
        C[(size_t)m * ldc + n] = silu_mul(v[0], v[1]);
    else
        C[(size_t)m * ldc + n] = v[0];
}

// The same sums where a norm follows: added to the residual in place (with the product's bias, where it has one), whose rows
// are normed as add_rmsnorm does, bit for bit, in one kernel instead of two and without the product's way through
// memory.  Bound by its start and the runs' bytes.  Microseconds of product and norm at 17 / 64 / 225 / 1,024 rows, as
// kernels of their own / so: 1,024 x 3,072 15.5 / 14.0, 18.1 / 16.2, 24.0 / 21.3, 54.2 / 48.8; 1,024 x 2,048 13.2 / 11.6,
// 15.2 / 13.3, 21.5 / 18.8, 41.9 / 38.7; 2,560 x 9,728 43.6 / 42.1, 47.9 / 45.8, 107 / 98, 301 / 294.
template <int CHUNKS>
__global__ void gemm_f32_add_runs_rmsnorm_kernel(const float* __restrict__ parts, const float* __restrict__ A,
                                                 const float* __restrict__ W, int M, int K, int lda, int ldw,
                                                 float* __restrict__ residual, const float* __restrict__ weight,
                                                 float* __restrict__ out, int hidden, float eps,
                                                 const float* __restrict__ bias) {
    __shared__ float scratch[16];
    const int m = blockIdx.x, nvec = hidden >> 2;
    const size_t stride = (size_t)M * hidden;
    f32x4* res = reinterpret_cast<f32x4*>(residual + (size_t)m * hidden);
    f32x4 val[CHUNKS], wt[CHUNKS];
    float ss = 0.f;
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) {
        const int i = threadIdx.x + c * blockDim.x;
        if (i < nvec) wt[c] = reinterpret_cast<const f32x4*>(weight)[i];
    }
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) {
        const int i = threadIdx.x + c * blockDim.x;
        if (i < nvec) {
            const float* p = parts + (size_t)m * hidden + 4 * i;
            f32x4 run[FRUNS];
#pragma unroll
            for (int r = 0; r < FRUNS; ++r) run[r] = *reinterpret_cast<const f32x4*>(p + r * stride);
            f32x4 v = res[i], d = run[0];
#pragma unroll
            for (int r = 1; r < FRUNS; ++r) d = r & 1 ? d - run[r] : d + run[r];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                v[j] += finite_or_wide(d[j], A + (size_t)m * lda, W + (size_t)(4 * i + j) * ldw, K);
                if (bias) v[j] += bias[4 * i + j];
            }
            res[i] = v;
            val[c] = v;
            ss += v[0] * v[0] + v[1] * v[1] + v[2] * v[2] + v[3] * v[3];
        }
    }
    ss = block_sum(ss, scratch);
    const float rrms = rsqrtf(ss / (float)hidden + eps);
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) {
        const int i = threadIdx.x + c * blockDim.x;
        if (i < nvec) {
            f32x4 y;
#pragma unroll
            for (int j = 0; j < 4; ++j) y[j] = val[c][j] * rrms * wt[c][j];
            reinterpret_cast<f32x4*>(out + (size_t)m * hidden)[i] = y;
        }
    }
}

// Up to FEW k: a thread a result, bound by the results (2,048 x 6,144 of 1 and 3 k 15 and 19 us; the kernel on the
// float32 instruction took 40 and 39).
__global__ __launch_bounds__(256) void gemm_f32_few_kernel(const float* __restrict__ A, const float* __restrict__ W,
                                                           float* __restrict__ C, int M, int N, int K, int lda,
                                                           int ldw, int ldc) {
    const int n = blockIdx.x * 256 + threadIdx.x;
    if (n >= N) return;
    double w[FEW];
#pragma unroll
    for (int k = 0; k < FEW; ++k) w[k] = k < K ? W[(size_t)n * ldw + k] : 0.f;
    for (int m = blockIdx.y; m < M; m += gridDim.y) {
        const float* a = A + (size_t)m * lda;
        double s = a[0] * w[0];
#pragma unroll
        for (int k = 1; k < FEW; ++k)
            if (k < K) s = fma((double)a[k], w[k], s);
        C[(size_t)m * ldc + n] = (float)s;
    }
}

// 16-row blocks of W of a product of N result columns
template <bool GLU>
static int w_blocks(int N) {
    return GLU ? (N + 7) / 8 : (N + 15) / 16;
}

template <int NT, bool GLU>
static int launch_stream(const float* A, const float* W, float* C, int M, int N, int K, int lda, int ldw,
                         int ldc, hipStream_t stream) {
    const int mt = M <= 16 ? 1 : 2;
    const dim3 grid((w_blocks<GLU>(N) + NT - 1) / NT, (M + 16 * mt - 1) / (16 * mt)), block(FRUNS * RL_WAVE);
    if (grid.y > 65535) return RL_ERR_ARG;
    if (mt == 1)
        hipLaunchKernelGGL((gemm_f32_stream_kernel<NT, 1, GLU>), grid, block, 0, stream, A, W, C, M, N, K, lda, ldw, ldc);
    else
        hipLaunchKernelGGL((gemm_f32_stream_kernel<NT, 2, GLU>), grid, block, 0, stream, A, W, C, M, N, K, lda, ldw, ldc);
    return rl_launch_status();
}

template <int TM, int TN, Length L, bool GLU>
static int launch_tile_of(const float* A, const float* W, float* C, float* parts, int M, int N, int K, int lda,
                       int ldw, int ldc, int groups, hipStream_t stream) {
    const int tm = (M + 32 * TM - 1) / (32 * TM);
    const dim3 block(256);
    if (groups == 1) {
        const int tn = (w_blocks<GLU>(N) + 2 * TN - 1) / (2 * TN);
        if ((long long)tm * tn > 0x7fffffffLL / 16) return RL_ERR_ARG;
        hipLaunchKernelGGL((gemm_f32_tile_kernel<TM, TN, L, false, GLU>), dim3(tm * tn), block, 0, stream, A, W, C, M, N,
                           K, lda, ldw, ldc, tm, tn, FRUNS);
        return rl_launch_status();
    }
    const int rows = GLU ? 2 * N : N, tn = (rows + 32 * TN - 1) / (32 * TN);  // (the runs are those of the plain product)
    if ((long long)tm * tn > 0x7fffffffLL / 16) return RL_ERR_ARG;
    if (!parts || M > 65535) return RL_ERR_ARG;
    hipLaunchKernelGGL((gemm_f32_tile_kernel<TM, TN, L, true, false>), dim3(tm * tn, groups), block, 0, stream, A, W, parts,
                       M, rows, K, lda, ldw, ldc, tm, tn, FRUNS / groups);
    if (int code = rl_launch_status()) return code;
    if (!C) return RL_OK;  // (rl_gemm_f32_add_rmsnorm adds them)
    hipLaunchKernelGGL(gemm_f32_add_runs_kernel<GLU>, dim3((N + 255) / 256, M), block, 0, stream, parts, A, W, C, M, rows,
                       K, lda, ldw, ldc);
    return rl_launch_status();
}

template <int TM, int TN, bool GLU = false>
static int launch_tile(const float* A, const float* W, float* C, float* parts, int M, int N, int K, int lda,
                       int ldw, int ldc, int groups, hipStream_t stream) {
    if (K % 4) return launch_tile_of<TM, TN, ELEMENTS, GLU>(A, W, C, parts, M, N, K, lda, ldw, ldc, groups, stream);
    if (K % FCH) return launch_tile_of<TM, TN, PIECES, GLU>(A, W, C, parts, M, N, K, lda, ldw, ldc, groups, stream);
    return launch_tile_of<TM, TN, WHOLE, GLU>(A, W, C, parts, M, N, K, lda, ldw, ldc, groups, stream);
}

template <int NT, int MT, bool GLU>
static int launch_runs_of(const float* A, const float* W, float* C, int M, int N, int K, int lda, int ldw, int ldc, hipStream_t stream) {
    const int tm = (M + 16 * MT - 1) / (16 * MT), tn = (w_blocks<GLU>(N) + NT - 1) / NT;
    if ((long long)tm * tn > 0x7fffffffLL / 16) return RL_ERR_ARG;
    hipLaunchKernelGGL((gemm_f32_runs_kernel<NT, MT, GLU>), dim3(tm * tn), dim3(FRUNS * RL_WAVE), 0, stream, A, W, C, M, N, K,
                       lda, ldw, ldc, tm, tn);
    return rl_launch_status();
}

template <bool GLU>
static int launch_runs(const float* A, const float* W, float* C, int M, int N, int K, int lda, int ldw, int ldc, int nt, int mt,
                       hipStream_t stream) {
    // whole units of 16 bytes are loaded; offsets are 32-bit, those of a tile's rows beyond the matrices too
    const long long limit = 0xffffffffll / 4;
    if (((uintptr_t)A | (uintptr_t)W) % 16 || (lda | ldw) % 4 || K % FCH || ((GLU ? 2ll : 1ll) * N + 256) * ldw > limit || (M + 256ll) * lda > limit) return RL_ERR_ARG;
#define RL_RUNS(NTV, MTV) \
    if (nt == NTV && mt == MTV) return launch_runs_of<NTV, MTV, GLU>(A, W, C, M, N, K, lda, ldw, ldc, stream)
    RL_RUNS(1, 1);
    RL_RUNS(2, 1);
    RL_RUNS(3, 1);
    RL_RUNS(6, 1);
    RL_RUNS(1, 2);
    RL_RUNS(2, 2);
    RL_RUNS(3, 2);
    RL_RUNS(4, 2);
    RL_RUNS(6, 2);
    RL_RUNS(2, 3);
    RL_RUNS(3, 3);
    RL_RUNS(4, 3);
    RL_RUNS(3, 4);
    RL_RUNS(4, 4);
    RL_RUNS(6, 4);
    RL_RUNS(4, 5);
#undef RL_RUNS
    return RL_ERR_ARG;
}

template <bool GLU>
static int launch_product(const float* A, const float* W, float* C, float* parts, int M, int N, int K, int lda,
                          int ldw, int ldc, int tile, int groups, hipStream_t stream) {
    if (tile <= 3) {
        if (groups != 1) return RL_ERR_ARG;
        if (tile == 1) return launch_stream<1, GLU>(A, W, C, M, N, K, lda, ldw, ldc, stream);
        if (tile == 2) return launch_stream<2, GLU>(A, W, C, M, N, K, lda, ldw, ldc, stream);
        if (tile == 3) return launch_stream<3, GLU>(A, W, C, M, N, K, lda, ldw, ldc, stream);
        return RL_ERR_ARG;
    }
    if (tile == 32) return launch_tile<1, 2, GLU>(A, W, C, parts, M, N, K, lda, ldw, ldc, groups, stream);
    if (tile == 64) return launch_tile<2, 2, GLU>(A, W, C, parts, M, N, K, lda, ldw, ldc, groups, stream);
    if (tile == 128) return launch_tile<4, 4, GLU>(A, W, C, parts, M, N, K, lda, ldw, ldc, groups, stream);
    return RL_ERR_ARG;
}

template <bool GLU>
static int launch_wide(const float* A, const float* W, float* C, void* pieces, int M, int N, int K, int lda,
                       int ldw, int ldc, int cols, hipStream_t stream) {
    const int chunks = K / FCH, blocks = (M + 15) / 16;
    if (!pieces || (uintptr_t)pieces % 16 || K <= 0 || K % FCH || lda < K || ldw < K || ldc < N || (cols != 128 && cols != 96))
        return RL_ERR_ARG;
    const int tm = (M + 255) / 256, tn = (w_blocks<GLU>(N) + cols / 16 - 1) / (cols / 16);
    // the pieces of a tile are addressed with 32 bits
    if (K > 1 << 20 || blocks > 65535 || (long long)tm * tn > 0x7fffffffLL / 16) return RL_ERR_ARG;
    hipLaunchKernelGGL(gemm_f32_pieces_kernel, dim3((chunks + 3) / 4, blocks), dim3(256), 0, stream, A, (__bf16*)pieces, M,
                       chunks, lda, (chunks + FRUNS - 1) / FRUNS);
    if (int code = rl_launch_status()) return code;
    if (cols == 128)
        hipLaunchKernelGGL((gemm_f32_wide_kernel<4, GLU>), dim3(tm * tn), dim3(512), 0, stream, A, (const __bf16*)pieces, W, C,
                           M, N, K, lda, ldw, ldc, tm, tn);
    else
        hipLaunchKernelGGL((gemm_f32_wide_kernel<3, GLU>), dim3(tm * tn), dim3(512), 0, stream, A, (const __bf16*)pieces, W, C,
                           M, N, K, lda, ldw, ldc, tm, tn);
    return rl_launch_status();
}

// Rows of A and W may be strided; the inner dimension is contiguous.  `tile`: 1, 2 and 3 stream the
// weights (so many tiles of 16 weight rows a workgroup), 32, 64 and 128 are the rows of A a tile takes;
// `groups` (1, 2, 4, 8): workgroups that share a tile's runs, with `parts` [8, M, N] for the runs' results
// where there is more than one.
extern "C" int rl_gemm_f32(const float* A, const float* W, float* C, float* parts, int M, int N, int K, int lda,
                           int ldw, int ldc, int tile, int groups, hipStream_t stream) {
    if (M <= 0 || N <= 0) return RL_OK;
    if (K <= 0 || lda < K || ldw < K || ldc < N || !C) return RL_ERR_ARG;
    if (groups != 1 && groups != 2 && groups != 4 && groups != 8) return RL_ERR_ARG;
    if (K <= FEW) {  // whatever the tile
        hipLaunchKernelGGL(gemm_f32_few_kernel, dim3((N + 255) / 256, M < 1024 ? M : 1024), dim3(256), 0, stream, A, W,
                           C, M, N, K, lda, ldw, ldc);
        return rl_launch_status();
    }
    return launch_product<false>(A, W, C, parts, M, N, K, lda, ldw, ldc, tile, groups, stream);
}

// The same with silu(gate) * up of the packed [gate | up] matrix W[2 N, K]; `parts` [8, M, 2 N].
extern "C" int rl_gemm_f32_gated(const float* A, const float* W, float* C, float* parts, int M, int N, int K, int lda,
                                 int ldw, int ldc, int tile, int groups, hipStream_t stream) {
    if (M <= 0 || N <= 0) return RL_OK;
    if (K <= FEW || lda < K || ldw < K || ldc < N || !C || N > 0x3fffffff) return RL_ERR_ARG;
    if (groups != 1 && groups != 2 && groups != 4 && groups != 8) return RL_ERR_ARG;
    return launch_product<true>(A, W, C, parts, M, N, K, lda, ldw, ldc, tile, groups, stream);
}

// The same for K a multiple of 32 and rows that begin with whole units of 16 bytes, a wave a run: a tile is 16 nt weight rows x
// 16 mt rows of A.
extern "C" int rl_gemm_f32_runs(const float* A, const float* W, float* C, int M, int N, int K, int lda, int ldw, int ldc, int nt,
                                int mt, hipStream_t stream) {
    if (M <= 0 || N <= 0) return RL_OK;
    if (K < FCH || lda < K || ldw < K || ldc < N || !A || !W || !C) return RL_ERR_ARG;
    return launch_runs<false>(A, W, C, M, N, K, lda, ldw, ldc, nt, mt, stream);
}

extern "C" int rl_gemm_f32_runs_gated(const float* A, const float* W, float* C, int M, int N, int K, int lda, int ldw, int ldc,
                                      int nt, int mt, hipStream_t stream) {
    if (M <= 0 || N <= 0) return RL_OK;
    if (K < FCH || lda < K || ldw < K || ldc < N || !A || !W || !C || N > 0x3fffffff) return RL_ERR_ARG;
    return launch_runs<true>(A, W, C, M, N, K, lda, ldw, ldc, nt, mt, stream);
}

// The same for many rows and K a multiple of 32: `pieces` holds 96 K bytes for every 16 rows of A; `cols` (128 or 96) are
// the rows of W a tile takes.
extern "C" int rl_gemm_f32_wide(const float* A, const float* W, float* C, void* pieces, int M, int N, int K, int lda,
                                int ldw, int ldc, int cols, hipStream_t stream) {
    if (M <= 0 || N <= 0) return RL_OK;
    return launch_wide<false>(A, W, C, pieces, M, N, K, lda, ldw, ldc, cols, stream);
}

extern "C" int rl_gemm_f32_wide_gated(const float* A, const float* W, float* C, void* pieces, int M, int N, int K, int lda,
                                      int ldw, int ldc, int cols, hipStream_t stream) {
    if (M <= 0 || N <= 0) return RL_OK;
    if (N > 0x3fffffff) return RL_ERR_ARG;
    return launch_wide<true>(A, W, C, pieces, M, N, K, lda, ldw, ldc, cols, stream);
}

// residual[M, N] += A W^T (+ bias) in place and out[M, N] = rmsnorm(residual) * weight, where f32_plan cuts the product into
// runs (`tile` 32, 64 or 128, `groups` 2, 4 or 8); N a multiple of 4 up to 16 K.
extern "C" int rl_gemm_f32_add_rmsnorm(const float* A, const float* W, float* parts, int M, int N, int K, int lda, int ldw,
                                       int tile, int groups, float* residual, const float* weight, float* out, float eps,
                                       const float* bias, hipStream_t stream) {
    if (M <= 0 || N <= 0) return RL_OK;
    if (K <= FEW || lda < K || ldw < K || N % 4 || N > 16 * 1024 || !parts || !residual || !weight || !out) return RL_ERR_ARG;
    if (groups != 2 && groups != 4 && groups != 8) return RL_ERR_ARG;
    int code = RL_ERR_ARG;
    if (tile == 32) code = launch_tile<1, 2>(A, W, nullptr, parts, M, N, K, lda, ldw, N, groups, stream);
    if (tile == 64) code = launch_tile<2, 2>(A, W, nullptr, parts, M, N, K, lda, ldw, N, groups, stream);
    if (tile == 128) code = launch_tile<4, 4>(A, W, nullptr, parts, M, N, K, lda, ldw, N, groups, stream);
    if (code != RL_OK) return code;
    // threads as for add_rmsnorm: the order of the row's sum
    const int threads = (N / 4 + RL_WAVE - 1) / RL_WAVE * RL_WAVE;
    if (threads <= 1024)
        hipLaunchKernelGGL(gemm_f32_add_runs_rmsnorm_kernel<1>, dim3(M), dim3(threads), 0, stream, parts, A, W, M, K, lda, ldw,
                           residual, weight, out, N, eps, bias);
    else
        hipLaunchKernelGGL(gemm_f32_add_runs_rmsnorm_kernel<4>, dim3(M), dim3(1024), 0, stream, parts, A, W, M, K, lda, ldw,
                           residual, weight, out, N, eps, bias);
    return rl_launch_status();
}
