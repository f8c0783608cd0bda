// Float32 matrix product C[M,N] = A[M,K] * W[N,K]^T on the matrix cores' bfloat16 instruction
// (v_mfma_f32_16x16x32_bf16), without the loss of a bfloat16 product: every float32 operand is
// split into three bfloat16 numbers that add up to it (24 bits of mantissa are 8 + 8 + 8, and the
// exponents are the same), and a product of two operands is the six partial products
//   hi hi + (hi mid + mid hi) + (mid mid + hi lo + lo hi),
// each exact before it is added up in float32.  The three left out are below 2^-26 of the product, less
// than the rounding of one float32 addition.  The float32 instruction (v_mfma_f32_16x16x4_f32) has 157
// TFLOP/s at most, and the kernel on it that this one replaces reached 101; six bfloat16 instructions
// come to a sixth of 2.5 PFLOP/s, of which the library's bfloat16 products reach half.  Measured at 2,048
// rows: 6,144 x 4,096 1,018 -> 530 us, 24,576 x 4,096 4,259 -> 2,000 us, 4,096 x 12,288 2,007 -> 985 us
// (200 to 210 TFLOP/s); at 225 rows of a small model 6,144 x 1,024 53 -> 36 us and 1,024 x 3,072 68 -> 20
// us.  Error against 64 bits over normal operands, relative to the result: K = 4,096 4.1e-7 -> 3.4e-7,
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
// What the split cannot represent is computed again without it: an element that comes out
// infinite or not a number (an infinite operand meets a zero piece of the other; an operand
// above bfloat16's largest number rounds to infinity) is the plain float32 sum instead.
//
// The transposed product is computed (W supplies the A operand, the rows of A the B operand),
// so a lane's four results are four consecutive n of one row of C.
#include "common.h"

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

#define FRUNS 8  // runs of K = waves per workgroup of the streaming kernel
#define FCH 32   // k per chunk

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

// `flip`: a sign bit to turn
__device__ inline Split split8(f32x4 x, f32x4 y, uint32_t flip = 0) {
    u32x4 p[3];
    float v[8];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const float lo = x[j], hi = y[j];
        v[j] = __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, lo) ^ flip);
        v[4 + j] = __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, hi) ^ flip);
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

// the element as it is, or the plain float32 sum where the split gave no finite number
__device__ inline float finite_or_plain(float v, const float* a, const float* w, int K) {
    if (__builtin_isfinite(v)) return v;
    float s = 0.f;
    for (int k = 0; k < K && s == s; ++k) s = fmaf(a[k], w[k], s);
    return s;
}

// four consecutive floats of a row, zeros beyond `limit` (elements left in the row)
template <bool VEC>
__device__ inline f32x4 load_k4(const float* p, int limit) {
    if (VEC) {
        if (limit >= 4) return *reinterpret_cast<const f32x4*>(p);
        return (f32x4){0.f, 0.f, 0.f, 0.f};  // VEC: K is a multiple of 4, a piece is whole or absent
    }
    f32x4 v;
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = i < limit ? p[i] : 0.f;
    return v;
}

// ---- up to 16 rows: the weights are streamed once -----------------------------------------------
// One workgroup per NT tiles of 16 rows of W, one wave per run of K.  Bound by the weights' bytes, and from a
// few rows on by the rows of A beside them, which every workgroup reads whole (f32_plan says when NT is 2 or 3).
template <int NT, bool VEC>
__global__ __launch_bounds__(FRUNS* RL_WAVE) void gemm_f32_stream_kernel(
    const float* __restrict__ A, const float* __restrict__ W, float* __restrict__ C, int M, int N,
    int K, int lda, int ldw, int ldc) {
    __shared__ float red[FRUNS][NT * 256];

    const int lane = threadIdx.x & (RL_WAVE - 1);
    const int wave = threadIdx.x / RL_WAVE;
    const int r16 = lane & 15;
    const int g = lane >> 4;
    const int n0 = blockIdx.x * NT * 16;

    // rows beyond the matrices read the last row; their results are dropped at the end
    const float* wrow[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) wrow[nt] = W + (size_t)min(n0 + nt * 16 + r16, N - 1) * ldw + 8 * g;
    const float* arow = A + (size_t)min(r16, M - 1) * lda + 8 * g;

    f32x4 acc[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) acc[nt] = (f32x4){0.f, 0.f, 0.f, 0.f};

    const int chunks = (K + FCH - 1) / FCH;
    const int per = (chunks + FRUNS - 1) / FRUNS;
    const int c_lo = min(chunks, wave * per), c_hi = min(chunks, c_lo + per);

    // two chunks are asked for together: 256 contiguous bytes of every row (with many tiles one, whose
    // loads are as many)
    constexpr int U = NT > 2 ? 1 : 2;
    struct Rows {
        f32x4 w[U][NT][2], a[U][2];
    };
    auto load_group = [&](int c, Rows& r) {  // whole chunks: no predicate
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
#pragma unroll
                for (int nt = 0; nt < NT; ++nt)
                    r.w[u][nt][h] = *reinterpret_cast<const f32x4*>(wrow[nt] + (c + u) * FCH + 4 * h);
                r.a[u][h] = *reinterpret_cast<const f32x4*>(arow + (c + u) * FCH + 4 * h);
            }
        // the loads stay here, in front of the other group's products (left to itself the
        // scheduler moves them down to their use and nothing is in flight during the products)
        __builtin_amdgcn_sched_barrier(0);
    };
    auto products = [&](const f32x4 (&w)[NT][2], const f32x4 (&a)[2]) {
        const Split as = split8(a[0], a[1], (wave & 1u) << 31);
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
                    acc[n0 + j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ws[j].p[PIECE_W[s]], as.p[PIECE_A[s]],
                                                                         acc[n0 + j], 0, 0, 0);
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
        const int whole = VEC ? min(c_hi, K / FCH) : c_lo;  // unaligned rows: every chunk is checked
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
        const int k = c * FCH + 8 * g;  // this lane's first k of the chunk
        f32x4 w[NT][2], a[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) w[nt][h] = load_k4<VEC>(wrow[nt] + c * FCH + 4 * h, K - k - 4 * h);
            a[h] = load_k4<VEC>(arow + c * FCH + 4 * h, K - k - 4 * h);
        }
        products(w, a);
    }

    // the runs are added in their order
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int i = 0; i < 4; ++i) red[wave][(nt * 4 + i) * 64 + lane] = acc[nt][i];
    __syncthreads();
    for (int e = threadIdx.x; e < NT * 256; e += FRUNS * RL_WAVE) {
        const int ln = e & 63;
        const int n = n0 + (e >> 8) * 16 + 4 * (ln >> 4) + ((e >> 6) & 3);
        const int m = ln & 15;
        if (n >= N || m >= M) continue;
        float v = red[0][e];
#pragma unroll
        for (int w = 1; w < FRUNS; ++w) v = w & 1 ? v - red[w][e] : v + red[w][e];
        C[(size_t)m * ldc + n] = finite_or_plain(v, A + (size_t)m * lda, W + (size_t)n * ldw, K);
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
template <int TM, int TN, bool FULL, bool RUNS>
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
        from_w[i] = W + (size_t)min(n0 + row, N - 1) * ldw + 8 * piece;
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
        const int k = c * FCH + 8 * piece;
        auto four = [&](const float* p, int h) {
            return FULL ? *reinterpret_cast<const f32x4*>(p) : load_k4<false>(p, K - k - 4 * h);
        };
#pragma unroll
        for (int h = 0; h < 2; ++h) {
#pragma unroll
            for (int i = 0; i < PA; ++i) r.a[i][h] = four(from_a[i] + c * FCH + 4 * h, h);
#pragma unroll
            for (int i = 0; i < PW; ++i) r.w[i][h] = four(from_w[i] + c * FCH + 4 * h, h);
        }
    };
    auto store = [&](const Raw& r, int buf) {
        const uint32_t flip = (stored & 1u) << 31;
        if (++next == (stored + 1) * per) ++stored;
#pragma unroll
        for (int i = 0; i < PA; ++i) {
            const Split s = split8(r.a[i][0], r.a[i][1], flip);
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
#pragma unroll
    for (int x = 0; x < TN; ++x)
#pragma unroll
        for (int y = 0; y < TM; ++y) {
            const int m = m0 + (wm + y) * 16 + r16, n = n0 + (wn + x) * 16 + 4 * g;
            if (m >= M) continue;
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (n + i < N)
                    C[(size_t)m * ldc + n + i] =
                        finite_or_plain(total[x][y][i], A + (size_t)m * lda, W + (size_t)(n + i) * ldw, K);
        }
}

// the runs of the tile kernel added in their order
__global__ __launch_bounds__(256) void gemm_f32_add_runs_kernel(
    const float* __restrict__ parts, const float* __restrict__ A, const float* __restrict__ W,
    float* __restrict__ C, int M, int N, int K, int lda, int ldw, int ldc) {
    const int m = blockIdx.y;
    const int n = blockIdx.x * 256 + threadIdx.x;
    if (n >= N) return;
    float v = parts[(size_t)m * N + n];
#pragma unroll
    for (int r = 1; r < FRUNS; ++r) {
        const float x = parts[((size_t)r * M + m) * N + n];
        v = r & 1 ? v - x : v + x;
    }
    C[(size_t)m * ldc + n] = finite_or_plain(v, A + (size_t)m * lda, W + (size_t)n * ldw, K);
}

template <int NT>
static int launch_stream(const float* A, const float* W, float* C, int M, int N, int K, int lda, int ldw,
                         int ldc, bool vec, hipStream_t stream) {
    dim3 grid((N + 16 * NT - 1) / (16 * NT)), block(FRUNS * RL_WAVE);
    if (vec)
        hipLaunchKernelGGL((gemm_f32_stream_kernel<NT, true>), grid, block, 0, stream, A, W, C, M, N, K,
                           lda, ldw, ldc);
    else
        hipLaunchKernelGGL((gemm_f32_stream_kernel<NT, false>), grid, block, 0, stream, A, W, C, M, N, K,
                           lda, ldw, ldc);
    return rl_launch_status();
}

template <int TM, int TN>
static int launch_tile(const float* A, const float* W, float* C, float* parts, int M, int N, int K, int lda,
                       int ldw, int ldc, int groups, bool full, hipStream_t stream) {
    const int tm = (M + 32 * TM - 1) / (32 * TM), tn = (N + 32 * TN - 1) / (32 * TN);
    if ((long long)tm * tn > 0x7fffffffLL / 16) return RL_ERR_ARG;
    const dim3 block(256);
    if (groups == 1) {
        const dim3 grid(tm * tn);
        if (full)
            hipLaunchKernelGGL((gemm_f32_tile_kernel<TM, TN, true, false>), grid, block, 0, stream, A, W, C, M,
                               N, K, lda, ldw, ldc, tm, tn, FRUNS);
        else
            hipLaunchKernelGGL((gemm_f32_tile_kernel<TM, TN, false, false>), grid, block, 0, stream, A, W, C, M,
                               N, K, lda, ldw, ldc, tm, tn, FRUNS);
        return rl_launch_status();
    }
    if (!parts || M > 65535) return RL_ERR_ARG;
    const dim3 grid(tm * tn, groups);
    if (full)
        hipLaunchKernelGGL((gemm_f32_tile_kernel<TM, TN, true, true>), grid, block, 0, stream, A, W, parts, M, N,
                           K, lda, ldw, ldc, tm, tn, FRUNS / groups);
    else
        hipLaunchKernelGGL((gemm_f32_tile_kernel<TM, TN, false, true>), grid, block, 0, stream, A, W, parts, M, N,
                           K, lda, ldw, ldc, tm, tn, FRUNS / groups);
    if (int code = rl_launch_status()) return code;
    hipLaunchKernelGGL(gemm_f32_add_runs_kernel, dim3((N + 255) / 256, M), block, 0, stream, parts, A, W, C, M, N,
                       K, lda, ldw, ldc);
    return rl_launch_status();
}

// Rows of A and W may be strided; the inner dimension is contiguous.  `tile`: 1, 2 and 3 stream the
// weights (up to 16 rows; so many tiles of 16 weight rows a workgroup), 32, 64 and 128 are the rows of A a tile takes;
// `groups` (1, 2, 4, 8): workgroups that share a tile's runs, with `parts` [8, M, N] for the runs' results
// where there is more than one.
extern "C" int rl_gemm_f32(const float* A, const float* W, float* C, float* parts, int M, int N, int K, int lda,
                           int ldw, int ldc, int tile, int groups, hipStream_t stream) {
    if (M <= 0 || N <= 0) return RL_OK;
    if (K <= 0 || lda < K || ldw < K || ldc < N) return RL_ERR_ARG;
    if (groups != 1 && groups != 2 && groups != 4 && groups != 8) return RL_ERR_ARG;
    const bool vec = K % 4 == 0 && lda % 4 == 0 && ldw % 4 == 0 &&
                     (reinterpret_cast<uintptr_t>(A) & 15) == 0 &&
                     (reinterpret_cast<uintptr_t>(W) & 15) == 0;
    const bool full = vec && K % FCH == 0;
    if (tile <= 3) {
        if (M > 16 || groups != 1) return RL_ERR_ARG;
        if (tile == 1) return launch_stream<1>(A, W, C, M, N, K, lda, ldw, ldc, vec, stream);
        if (tile == 2) return launch_stream<2>(A, W, C, M, N, K, lda, ldw, ldc, vec, stream);
        if (tile == 3) return launch_stream<3>(A, W, C, M, N, K, lda, ldw, ldc, vec, stream);
        return RL_ERR_ARG;
    }
    if (tile == 32) return launch_tile<1, 2>(A, W, C, parts, M, N, K, lda, ldw, ldc, groups, full, stream);
    if (tile == 64) return launch_tile<2, 2>(A, W, C, parts, M, N, K, lda, ldw, ldc, groups, full, stream);
    if (tile == 128) return launch_tile<4, 4>(A, W, C, parts, M, N, K, lda, ldw, ldc, groups, full, stream);
    return RL_ERR_ARG;
}
