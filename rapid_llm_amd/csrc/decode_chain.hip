// All layers of a decode step of up to 16 single tokens in one launch (bfloat16, heads of 128 channels): the
// products of gemm_bf16.hip and the decode attention of attention_mfma.hip as one chain of items.
//
// What bounds a decode step of few tokens over small matrices is not the weights' bytes but what every kernel of a dependent
// chain costs beside them: 3.5 us of start, first loads and tail, six kernels a layer, with nothing of one kernel beside the next.  Here
// one workgroup a compute unit stays for the whole step.  An item is a tile of 16 weight rows (a pair of gate
// and up tiles), or a request's kv head and a share of its keys.  While the items of one phase are finished and the next
// phase's input travels, the weights of the next phase (and the keys of the next attention) are on their way
// already: they depend on nothing.
//
// Items are numbered in the order of their dependencies and dealt to the workgroups in turn.  That needs every workgroup that
// has items to be running, whatever else the chip does: a workgroup enters its name when it starts; when all have, or
// after some time, the list is closed, the items are dealt to those on it, and a workgroup that starts later leaves at once.
// (Waits are bounded all the same: a workgroup that runs into the bound ends the launch, the step's result is NaN, every
// later launch ends at once, and a word in host memory says so.)
//
// A workgroup is eight waves that stream and multiply, and two that do what would stand in their way, because a
// wave's loads return in order: one waits for other workgroups' results and prepares the attention's queries and the norms'
// factors, one adds the waves' partial sums and stores results.  Weights and rows of X go from memory straight into LDS,
// a ring of chunks a wave.  The waves meet through counters in LDS, there is no barrier.  A unit answers its waves' requests
// in order, so a phase's weights are asked for when the phase before has stored its results: asked for at once, they kept the
// stores and everything that other workgroups' results are looked for with waiting (one row of Qwen3-0.6B 852 against
// 808 us a step, where six kernels a layer take 988; two 945 against 860 and 1,032).
//
// What one workgroup writes and another reads inside the launch passes by the dies' L2 caches: agent-scope stores and
// loads.  Two ways to know that it is there:
//   * TAGGED (one row or two): every 4 bytes of result travel with the launch's number in one 8-byte store, and who needs
//     them asks for them until the number is right: one trip through memory, 1.3 to 1.5 us a phase where storing,
//     waiting for the stores, a flag, seeing it and loading are 2.1 to 2.3 (256 workgroups, nothing else going on).  No
//     place is written twice in a launch.
//   * otherwise a workgroup stores, waits until that has reached memory and then says up to which phase of which launch it is done, in a
//     line of its own (flags side by side in lines: 3.2 to 4.0 us a phase; stores to one line follow each other).  Rows of
//     the products' inputs are then read through the L2: a line of them has one writer, who has written all of it, and
//     nobody has asked for it before.
#include "common.h"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32;
typedef unsigned long long u64;
typedef u32 u32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void* rl_lds_ptr;

#define D 128                // channels of a head
#define SW 8                 // waves that stream
#define CH_WAVES 10          // and with the two others
#define CH_THREADS (CH_WAVES * RL_WAVE)
#define KSTEP 128            // k elements of a chunk: 16 rows of 256 bytes
#define W_CHUNK 4096
#define CH_MAX_GROUP 4       // query heads a kv head
#define CH_MAX_ROWS 16
#define CH_TAGGED_ROWS 2     // rows up to which results travel with the launch's number
#define CH_KEYS (32 * SW)    // keys that the waves walk in one step
#define CH_ALONE (2 * CH_KEYS)  // keys up to which a request's context is one share
#define CH_MAX_WORKGROUPS 512
#define FLAG_STRIDE 8        // words of 64 bits between two workgroups' flags
#define PHASES 5
#define AUX_SC1 16           // a load that passes by this die's L2

#define RL_CONSTANT __attribute__((address_space(4)))  // read by scalar loads

enum Phase { PH_QKV, PH_ATT, PH_O, PH_GU, PH_DOWN };

// of a layer; next_norm is that of the layer behind (null: the last one's product is stored as it is)
struct ChainLayer {
    const bf16_t *w_qkv, *w_o, *w_gu, *w_down;
    const float *q_norm, *k_norm, *ff_norm, *next_norm;
    bf16_t *k_pages, *v_pages;
};

// what the workgroups of a launch know of each other; zeros before the first launch
#define LIST_CLOSED 0x80000000u
// The number of the last launch before they begin again at 0: tags, a launch's number + 1, are never 0, which lies where nobody
// has stored yet.  When it ends, everything that holds tags is cleared, so that none is met a second time.
#define LAST_LAUNCH 0xfffffffeu
struct Control {
    u32 list;      // workgroups that have entered their names
    u32 pad0[31];
    u64 dealt;     // launch + 1, workgroups on the list
    u32 pad1[30];
    u32 left;      // workgroups that have ended
    u32 launch;
    u32 abort;     // of a launch that was given up: every later one ends at once
    u32 pad2[29];
    u64 flags[CH_MAX_WORKGROUPS * FLAG_STRIDE];  // phases that a workgroup is done with, and the tag of the launch that they are of
};
// Whether a workgroup's flag says that it is done with so many phases of the launch.  A flag names its launch: launches
// that write none pass between two that do, any number of them, and a flag that was never written names none.
__device__ __host__ inline bool done_with(u64 flag, u32 tag, u32 phases) { return (u32)(flag >> 32) == tag && (u32)flag >= phases; }

// n / d for n below 2^32 / d: a multiplication
struct Divisor {
    u32 d, inverse;
    __host__ void set(u32 by) { d = by, inverse = (u32)((0x100000000ull + by - 1) / by); }
};

struct ChainArgs {
    const RL_CONSTANT ChainLayer* layers;
    const bf16_t* x;    // [M, H] the first layer's normed rows
    float* residual;    // [M, H]
    bf16_t* out;        // [M, H] the last layer's product
    const int *positions, *token_slot, *block_table;
    const float *cos_tab, *sin_tab;
    unsigned char* space;   // a layer's rows and sums, layer_bytes each
    u64* shares;            // the attention's shares: numbers with the launch's
    Control* control;
    u64* tagged;            // the space of steps of few rows, and how many words of it and of the shares hold tags
    u64 tagged_words, share_words;
    u32* notice;            // in host memory: set by a launch that is given up
    int num_layers, M, H, nq, nkv, I, table_stride, page_size, nsplit;
    float scale_log2, qk_eps, norm_eps, ff_eps;
    // in a layer's space (the packed rows are at 0); at_res: the stream behind the output product (tagged)
    u32 layer_bytes, at_att, at_xt_ff, at_part_ff, at_act, at_xt, at_part, at_res, at_res_down;
    int n[PHASES];             // items of the phases of a layer
    Divisor per_layer, by_heads, by_rows, by_page;  // items of a layer, kv heads, rows, tokens a page
    u32 total;          // items of the launch
};
typedef const RL_CONSTANT ChainArgs* Args;
// The arguments are read where they are used (a scalar load that finds them in its cache): kept in registers from the
// launch's beginning they are more than there are.
__device__ __forceinline__ Args fresh(Args a) {
    asm volatile("" : "+s"(a));
    return a;
}
// (and what follows from the lane is computed where it is used)
__device__ __forceinline__ int fresh(int lane) {
    asm volatile("" : "+v"(lane));
    return lane;
}

__device__ __forceinline__ u32 divide(u32 n, u32 inverse) { return inverse ? __umulhi(n, inverse) : n; }  // (1: 2^32)

struct Item {
    int phase, layer, idx;
};

template <typename T>
__device__ __forceinline__ T agent_load(const T* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T>
__device__ __forceinline__ void agent_store(T* p, T v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// two numbers rounded to bfloat16 (to nearest, ties to even), and back
__device__ __forceinline__ u32 pack_bf16(float a, float b) {
    return __builtin_bit_cast(u32, __builtin_convertvector((f32x2){a, b}, bf16x2));
}
__device__ __forceinline__ float low_bf16(u32 v) { return __uint_as_float(v << 16); }
__device__ __forceinline__ float high_bf16(u32 v) { return __uint_as_float(v & 0xffff0000u); }
__device__ __forceinline__ u64 pair64(u32 low, u32 high) { return (u64)low | (u64)high << 32; }
// every store of this wave has reached memory
__device__ __forceinline__ void stores_done() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// Counters in LDS.  In the streaming waves every access to LDS is written as an instruction: the compiler would wait for all
// loads on their way into LDS in front of it.
__device__ __forceinline__ u32 lds_at(const volatile void* p) { return (u32)(uintptr_t)(rl_lds_ptr)p; }
__device__ __forceinline__ u32 lds_get(const volatile void* p) {
    u32 v;
    asm volatile("ds_read_b32 %0, %1\n s_waitcnt lgkmcnt(0)" : "=&v"(v) : "v"(lds_at(p)) : "memory");
    return __builtin_amdgcn_readfirstlane(v);
}
// what this wave has read from and written to LDS is done before the counter changes
__device__ __forceinline__ void lds_put(volatile u32* p, u32 v) {
    asm volatile("s_waitcnt lgkmcnt(0)\n ds_write_b32 %0, %1" ::"v"(lds_at(p)), "v"(v) : "memory");
}
__device__ __forceinline__ void lds_count(volatile u32* p) {
    asm volatile("s_waitcnt lgkmcnt(0)\n ds_add_u32 %0, %1" ::"v"(lds_at(p)), "v"(1u) : "memory");
}

// sum over the lanes l, l + 16, l + 32, l + 48, left in all four
__device__ __forceinline__ float sum_rows_of_16(float v) {
    const unsigned u = __float_as_uint(v);
    const auto a = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    const unsigned w = __float_as_uint(__uint_as_float(a[0]) + __uint_as_float(a[1]));
    const auto b = __builtin_amdgcn_permlane16_swap(w, w, false, false);
    return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}
__device__ __forceinline__ float max_rows_of_16(float v) {
    const unsigned u = __float_as_uint(v);
    const auto a = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    const unsigned w = __float_as_uint(fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1])));
    const auto b = __builtin_amdgcn_permlane16_swap(w, w, false, false);
    return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}

// at most n of this wave's newest loads may still be on their way
__device__ __forceinline__ void wait_loads(int n) {
#define RL_WAIT(N) \
    case N: asm volatile("s_waitcnt vmcnt(" #N ")" ::: "memory"); break;
    switch (n < 16 ? n : 16) {
        RL_WAIT(0) RL_WAIT(1) RL_WAIT(2) RL_WAIT(3) RL_WAIT(4) RL_WAIT(5) RL_WAIT(6) RL_WAIT(7) RL_WAIT(8)
        RL_WAIT(9) RL_WAIT(10) RL_WAIT(11) RL_WAIT(12) RL_WAIT(13) RL_WAIT(14) RL_WAIT(15)
        default: asm volatile("s_waitcnt vmcnt(16)" ::: "memory"); break;
    }
#undef RL_WAIT
}

// 256 contiguous bytes a row: four pieces 64 bytes apart
__device__ __forceinline__ void ds_read_row(bf16x8 (&r)[4], u32 at) {
    asm volatile(
        "ds_read_b128 %0, %4\n ds_read_b128 %1, %4 offset:64\n ds_read_b128 %2, %4 offset:128\n ds_read_b128 %3, %4 offset:192\n"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(r[0]), "=&v"(r[1]), "=&v"(r[2]), "=&v"(r[3])
        : "v"(at)
        : "memory");
}
// a lane's four 16-byte units of a row, which lie at at ^ 16 j
__device__ __forceinline__ void ds_read4(bf16x8 (&r)[4], u32 at) {
    asm volatile(
        "ds_read_b128 %0, %4\n ds_read_b128 %1, %5\n ds_read_b128 %2, %6\n ds_read_b128 %3, %7\n"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(r[0]), "=&v"(r[1]), "=&v"(r[2]), "=&v"(r[3])
        : "v"(at), "v"(at ^ 16), "v"(at ^ 32), "v"(at ^ 48)
        : "memory");
}

// 128 bytes from each of g's places: the tagged pairs of a lane's 32 numbers of a row
__device__ __forceinline__ void ds_read_tagged(u32x4 (&r)[8], u32 at) {
    asm volatile(
        "ds_read_b128 %0, %8\n ds_read_b128 %1, %8 offset:16\n ds_read_b128 %2, %8 offset:32\n ds_read_b128 %3, %8 offset:48\n"
        "ds_read_b128 %4, %8 offset:64\n ds_read_b128 %5, %8 offset:80\n ds_read_b128 %6, %8 offset:96\n ds_read_b128 %7, %8 offset:112\n"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(r[0]), "=&v"(r[1]), "=&v"(r[2]), "=&v"(r[3]), "=&v"(r[4]), "=&v"(r[5]), "=&v"(r[6]), "=&v"(r[7])
        : "v"(at)
        : "memory");
}
// four 16-byte units, STRIDE bytes apart
template <int STRIDE>
__device__ __forceinline__ void ds_read_units(bf16x8 (&r)[4], u32 at) {
    asm volatile(
        "ds_read_b128 %0, %4\n ds_read_b128 %1, %4 offset:%5\n ds_read_b128 %2, %4 offset:%6\n ds_read_b128 %3, %4 offset:%7\n"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(r[0]), "=&v"(r[1]), "=&v"(r[2]), "=&v"(r[3])
        : "v"(at), "n"(STRIDE), "n"(2 * STRIDE), "n"(3 * STRIDE)
        : "memory");
}

// LDS of a workgroup.  XG: groups of four rows of X (0: one row, 1: up to 4 rows, 2: up to 8, 4: up to 16).
template <int XG>
struct Shape {
    static constexpr int XR = XG ? 4 * XG : 1;               // rows of X
    static constexpr int MP = XG ? 4 * XG : 4;               // rows that partial sums are kept of
    static constexpr int SLOT = W_CHUNK + (XG ? XG * 1024 : 512);
    static constexpr int DEPTH = XG == 0 ? 4 : XG == 4 ? 2 : 3;  // chunks of a wave's ring
    static constexpr int RING = DEPTH * SLOT;
    static constexpr int RED = SW * 2 * 4 * 4 * MP * 4;      // partial sums of eight waves, two tiles
    static constexpr int STATE = CH_MAX_GROUP * (D + 2);     // numbers of a wave's state of an attention item: in its ring's last slot
    static constexpr int AT_STATE = (DEPTH - 1) * SLOT;
    static constexpr int STAGE = (CH_MAX_GROUP + 2) * D * 2;     // prepared queries, the new key and value
    static constexpr int CTL = 512;
    static constexpr int AT_SCRATCH = SW * RING, AT_STAGE = AT_SCRATCH + RED, AT_CTL = AT_STAGE + STAGE;
    static constexpr int BYTES = AT_CTL + CTL;
    static_assert(STATE * 4 <= SLOT, "a state fits");
};

struct Ctl {
    u32 ready[2];     // items whose inputs are there, and whether the launch is over
    u32 summed[2];    // items whose partial sums have been read
    u32 streamed[2];  // items a wave is done with, over all eight waves
    u32 scaled[2];    // items whose norm's factors (whose token's own score) are there
    u32 stored[2];    // items whose results have been stored, and the one behind them has what it needs from memory
    u32 rank, workgroups, launch;
    float scale[CH_MAX_ROWS];
    float own[CH_MAX_GROUP];  // scores of the token's own key
    int pos[CH_MAX_ROWS], slot[CH_MAX_ROWS], run[CH_MAX_ROWS], shares[CH_MAX_ROWS];  // of the requests
};

__device__ __forceinline__ Item item_of(Args a, u32 t) {
    Item it;
    it.layer = divide(t, a->per_layer.inverse);
    it.idx = t - it.layer * a->per_layer.d;
    it.phase = 0;
#pragma unroll
    for (int p = 0; p < PHASES - 1; ++p)
        if (it.phase == p && it.idx >= a->n[p]) it.idx -= a->n[p], it.phase = p + 1;
    return it;
}

// A share of a request's keys.  The token's own key is apart from them: nobody has written it yet.
struct Share {
    int seq, hk, split, pos, lo, hi, shares;
    __device__ __forceinline__ Share(Args a, const Ctl* ctl, int idx) {
        const u32 r = divide(idx, a->by_heads.inverse);
        hk = idx - r * a->nkv;
        split = divide(r, a->by_rows.inverse);
        seq = r - split * a->M;
        pos = (int)lds_get(&ctl->pos[seq]);
        shares = (int)lds_get(&ctl->shares[seq]);
        const int run = (int)lds_get(&ctl->run[seq]);
        lo = split * run;
        hi = min(pos + 1, lo + run);
    }
    __device__ __forceinline__ bool empty() const { return split >= shares; }
    __device__ __forceinline__ bool own() const { return pos >= lo && pos < hi; }
};

// A wait in LDS; false: the launch is over.  Bounded by its turns (seconds of a wave that runs).
#define LDS_TURNS (1u << 24)
#define FLAG_TURNS (1u << 21)
#define LIST_TURNS 256u  // of a wait for workgroups that have not started, a few hundred microseconds in all
__device__ __forceinline__ void end_launch(Ctl* ctl) {
    lds_put(&ctl->ready[1], 1u);
    lds_put(&ctl->summed[1], 1u);
    lds_put(&ctl->streamed[1], 1u);
    lds_put(&ctl->scaled[1], 1u);
    lds_put(&ctl->stored[1], 1u);
}
__device__ __forceinline__ bool lds_wait(const u32* p, u32 least, Ctl* ctl) {
    for (u32 turns = 0;; ++turns) {
        u64 v;
        asm volatile("ds_read_b64 %0, %1\n s_waitcnt lgkmcnt(0)" : "=&v"(v) : "v"(lds_at(p)) : "memory");
        const u32 count = __builtin_amdgcn_readfirstlane((u32)v), over = __builtin_amdgcn_readfirstlane((u32)(v >> 32));
        if (over) return false;
        if ((int)(count - least) >= 0) return true;
        if (turns > LDS_TURNS) {
            end_launch(ctl);
            return false;
        }
    }
}
// one more turn of a wait for other workgroups; false: the launch is over
__device__ __forceinline__ bool turn(Args a, Ctl* ctl, u32& turns) {
    if ((++turns & 63) == 0) {
        if (lds_get(&ctl->ready[1])) return false;
        if (turns > FLAG_TURNS || __builtin_amdgcn_readfirstlane(agent_load(&a->control->abort))) {
            end_launch(ctl);
            return false;
        }
    }
    return true;
}

// N words of memory that carry the launch's number, asked for until all do.  at(i): word i's place; on(i): wanted
template <int N, typename At, typename On>
__device__ __forceinline__ bool tagged(u64 (&v)[N], Args a, Ctl* ctl, u32 tag, At at, On on) {
    u32 turns = 0;
    for (;;) {
#pragma unroll
        for (int i = 0; i < N; ++i) v[i] = on(i) ? agent_load(at(i)) : pair64(0, tag);
        bool late = false;
#pragma unroll
        for (int i = 0; i < N; ++i) late = late || (u32)(v[i] >> 32) != tag;
        if (!__any(late)) return true;
        __builtin_amdgcn_s_sleep(8);  // (so many waves that ask without a pause are in the answers' way)
        if (!turn(a, ctl, turns)) return false;
    }
}

// --------------------------------------------------------------------------------------------- //
// the waves that stream
// --------------------------------------------------------------------------------------------- //
template <int XG, bool TAGGED>
struct Streamer {
    using S = Shape<XG>;
    struct Source {  // an item's weights and rows
        const char *w, *x;
        u64 up;       // bytes from a gate tile to its up tile
        u32 k;
        int count;    // chunks of this wave, a pair's two counted apart
        int phase;
        bool pair, plain, l2, ok;  // plain: X is [M, K] as other kernels leave it; l2: X is read through the L2
    };
    Args args;
    unsigned char* lds;
    Ctl* ctl;
    const int lane, wave;
    u32 ring;          // LDS address of the wave's ring
    unsigned char* ring_ptr;
    u32 unit, w_at;    // the lane's places: its unit of a load's first row, of operands in a slot
    u32 issued = 0;    // loads asked for, all in all
    u32 need = 0;      // a byte a slot: loads asked for when the slot's chunk was complete
    int head = 0, tail = 0, held = 0;  // the ring
    Source is, next;   // the item whose chunks are being asked for, and the one behind it
    int is_seq = 0, is_entry = 0, pend = 0;  // pend: chunks whose X has not been asked for
    bool is_ready = false;  // its X may be asked for
    int next_seq = -1;
    u32 guard = 0;     // items whose states must have been read before the ring's last slot is written
    u32 rows, rank, workgroups, tag;

    __device__ __forceinline__ Streamer(Args a_, unsigned char* lds_, Ctl* ctl_, int wave_)
        : args(a_), lds(lds_), ctl(ctl_), lane(threadIdx.x & 63), wave(wave_) {
        const int r16 = lane & 15, g = lane >> 4;
        ring_ptr = lds + wave * S::RING;
        ring = lds_at(ring_ptr);
        rows = (u32)a_->M, rank = lds_get(&ctl_->rank), workgroups = lds_get(&ctl_->workgroups);
        tag = lds_get(&ctl_->launch) + 1;
        // A row's sixteen 16-byte units are permuted (unit u of row r at u ^ r): reads meet every bank once.
        unit = (u32)((r16 ^ g) * 16);
        w_at = (u32)(r16 * 256 + (((4 * g) ^ r16) * 16));
        is.ok = next.ok = false;
    }

    __device__ __forceinline__ static int chunks_of(int k, int wave) { return (k / KSTEP - wave + SW - 1) / SW; }

    __device__ __forceinline__ Source source(const Item& it) const {
        const Args a = fresh(args);
        const RL_CONSTANT ChainLayer& L = a->layers[it.layer];
        unsigned char* mine = a->space + (size_t)it.layer * a->layer_bytes;
        Source s;
        const bf16_t* w;
        int k;
        s.pair = it.phase == PH_GU, s.phase = it.phase;
        s.plain = it.phase == PH_QKV && it.layer == 0;
        s.l2 = !TAGGED && it.phase != PH_O;  // (rows of the attention: a line has a writer a request)
        if (it.phase == PH_QKV) {
            w = L.w_qkv, k = a->H;
            s.x = s.plain ? (const char*)a->x : (const char*)(mine - a->layer_bytes + a->at_xt);
        } else if (it.phase == PH_O) {
            w = L.w_o, k = a->nq * D, s.x = (const char*)(mine + a->at_att);
        } else if (it.phase == PH_GU) {
            w = L.w_gu, k = a->H, s.x = (const char*)(mine + a->at_xt_ff);
        } else {
            w = L.w_down, k = a->I, s.x = (const char*)(mine + a->at_act);
        }
        s.k = (u32)k;
        s.w = (const char*)w + (size_t)it.idx * 16 * k * 2;
        s.up = (u64)a->I * k * 2;
        s.count = chunks_of(k, wave) << (s.pair ? 1 : 0);
        s.ok = true;
        return s;
    }
    __device__ __forceinline__ void look_ahead(int seq) {
        const u32 t = rank + (u32)(seq + 1) * workgroups;
        const Args a = fresh(args);
        next.ok = false, next_seq = seq + 1;
        if (t >= a->total) return;
        const Item it = item_of(a, t);
        if (it.phase != PH_ATT) next = source(it);
    }
    __device__ __forceinline__ void begin(const Source& s, int seq) {
        is = s;
        is_seq = seq, is_entry = 0, is_ready = false;
    }

    __device__ __forceinline__ u32 chunk(const Source& s, int entry) const { return (u32)(wave + SW * (s.pair ? entry >> 1 : entry)); }
    __device__ __forceinline__ void mark(int slot) { need = (need & ~(0xffu << (8 * slot))) | ((issued & 0xffu) << (8 * slot)); }
    __device__ __forceinline__ void ask_x(const Source& s, int slot, int entry) {
#if defined(__HIP_DEVICE_COMPILE__)
        if (!(s.pair && (entry & 1))) {
            const int ln = fresh(lane);
            unsigned char* to = ring_ptr + slot * S::SLOT + W_CHUNK;
            if (s.plain) {  // into the layout of the others: 8 numbers of every row side by side
                auto rs = __builtin_amdgcn_make_buffer_rsrc((void*)s.x, 0, rows * s.k * 2, 0x00020000);
#pragma unroll
                for (int i = 0; i < (XG ? XG : 1); ++i) {
                    const u32 u = (u32)(64 * i + ln), m = u % S::XR;
                    if (XG || ln < 16)
                        __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (rl_lds_ptr)(to + i * 1024), 16, (m < rows ? m : 0u) * (s.k * 2) + u / S::XR * 16, chunk(s, entry) * 256, 0, 0);
                }
                issued += XG ? XG : 1;
            } else if (TAGGED) {  // [chunk][row][64 pairs of numbers, each with the launch's]
                auto rs = __builtin_amdgcn_make_buffer_rsrc((void*)s.x, 0, rows * s.k * 4, 0x00020000);
                if (XG || ln < 32)
                    __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (rl_lds_ptr)to, 16, ((u32)ln & (rows * 32 - 1)) * 16, chunk(s, entry) * (rows * 512), 0, AUX_SC1);
                issued += 1;
            } else {
                auto rs = __builtin_amdgcn_make_buffer_rsrc((void*)s.x, 0, S::XR * s.k * 2, 0x00020000);
#pragma unroll
                for (int i = 0; i < XG; ++i) {
                    if (s.l2)
                        __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (rl_lds_ptr)(to + i * 1024), 16, (u32)ln * 16, chunk(s, entry) * (S::MP * 256) + i * 1024, 0, 0);
                    else
                        __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (rl_lds_ptr)(to + i * 1024), 16, (u32)ln * 16, chunk(s, entry) * (S::MP * 256) + i * 1024, 0, AUX_SC1);
                }
                issued += XG;
            }
        }
        mark(slot);
#endif
    }
    __device__ __forceinline__ void ask_w(int slot, int entry) {
#if defined(__HIP_DEVICE_COMPILE__)
        const int g = fresh(lane) >> 4;
        const char* base = is.w + (is.pair && (entry & 1) ? is.up : 0);
        auto rs = __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, 16u * is.k * 2, 0x00020000);
        const u32 kb = chunk(is, entry) * (KSTEP * 2), row = (u32)g * (is.k * 2);
#pragma unroll
        for (int j = 0; j < 4; ++j)  // rows 4 j .. + 3
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (rl_lds_ptr)(ring_ptr + slot * S::SLOT + j * 1024), 16, row + (unit ^ (64 * j)), kb + j * 8 * is.k, 0, 0);
        issued += 4;
#endif
    }
    // Ask for what fits into the ring, of the item worked on (cur) and the one behind it.
    __device__ __forceinline__ void pump(int cur) {
        for (;;) {
            if (is_entry == is.count) {
                if (is_seq > cur || pend || !next.ok || next.phase != is.phase) return;
                begin(next, cur + 1);
                next.ok = false;
                continue;
            }
            if (held == S::DEPTH) return;
            if (head == S::DEPTH - 1 && guard) {
                if ((int)(lds_get(&ctl->summed[0]) - guard) < 0) return;
                guard = 0;
            }
            ask_w(head, is_entry);
            if (is_ready)
                ask_x(is, head, is_entry);
            else
                ++pend;
            head = head + 1 == S::DEPTH ? 0 : head + 1;
            ++is_entry;
            ++held;
        }
    }
    // X of the item worked on is there (TAGGED: may be)
    __device__ __forceinline__ void ask_pending() {
        int slot = head - pend, entry = is_entry - pend;
        if (slot < 0) slot += S::DEPTH;
        for (; pend; --pend, ++entry) {
            ask_x(is, slot, entry);
            slot = slot + 1 == S::DEPTH ? 0 : slot + 1;
        }
        is_ready = true;
    }
    __device__ __forceinline__ void wait_chunk() { wait_loads((int)((issued - (need >> (8 * tail))) & 0xffu)); }

    // X's operands of a chunk; true: some of it is not this launch's yet
    __device__ __forceinline__ bool read_x(bf16x8 (&x)[4], int slot, bool plain) {
        const int ln = fresh(lane), r16 = ln & 15, g = ln >> 4;
        const u32 at = ring + slot * S::SLOT + W_CHUNK;
        if (!TAGGED || plain) {
            ds_read_units<S::XR * 16>(x, at + (u32)((4 * g) * S::XR + (r16 & (S::XR - 1))) * 16);
            return false;
        }
        u32x4 r[8];
        ds_read_tagged(r, at + (r16 & (rows - 1)) * 512 + g * 128);
        u32 late = 0;
#pragma unroll
        for (int i = 0; i < 8; ++i) late |= (r[i][1] ^ tag) | (r[i][3] ^ tag);
#pragma unroll
        for (int j = 0; j < 4; ++j)
            x[j] = __builtin_bit_cast(bf16x8, (u32x4){r[2 * j][0], r[2 * j][2], r[2 * j + 1][0], r[2 * j + 1][2]});
        return __any(late != 0);
    }
    __device__ __forceinline__ static int behind(int slot, int by) {
        slot += by;
        return slot >= S::DEPTH ? slot - S::DEPTH : slot;
    }
    // the X of an item's chunks in the ring once more: from entry on, at the ring's end
    __device__ __forceinline__ bool ask_again(const Source& s, int entry, u32& turns) {
        const Args a = fresh(args);
        if (!turn(a, ctl, turns)) return false;
        __builtin_amdgcn_s_sleep(8);
        int slot = tail;
        for (int e = entry; e < s.count && e - entry < held; ++e) {
            ask_x(s, slot, e);
            slot = behind(slot, 1);
        }
        wait_loads(0);
        return true;
    }

    __device__ __forceinline__ void put_sums(const f32x4& v, int nt) {
        const int ln = fresh(lane), r16 = ln & 15, g = ln >> 4;
        if (r16 < S::MP) {
            const u32 at = lds_at(lds + S::AT_SCRATCH) + (u32)(((wave * 2 + nt) * 4 + g) * S::MP + r16) * 16;
            asm volatile("ds_write_b128 %0, %1" ::"v"(at), "v"(v) : "memory");
        }
    }

    // false: the launch is over
    __device__ __forceinline__ bool product(int seq, const Item& it) {
        if (is_seq != seq || !is.ok) {  // (else some of it is on its way already)
            // A unit answers its waves' requests in order: what the item before stores, and what its sums wait for, comes
            // before the next phase's weights.
            if (!lds_wait(ctl->stored, seq, ctl)) return false;
            if (next.ok && next_seq == seq)
                begin(next, seq);
            else
                begin(source(it), seq);
        }
        next.ok = false;
        const Source cur = is;
        const bool pair = cur.pair, plain = cur.plain;
        const int n = cur.count;
        pump(seq);
        if (guard) {
            if (!lds_wait(ctl->summed, guard, ctl)) return false;
            guard = 0;
            pump(seq);
        }
        const bool small = n <= S::DEPTH;  // all of it is in the ring
        if (TAGGED && (!small || plain)) ask_pending();
        look_ahead(seq);
        if (!TAGGED) {
            if (!lds_wait(ctl->ready, seq + 1, ctl)) return false;
            ask_pending();
        }
        f32x4 acc0 = {0.f, 0.f, 0.f, 0.f}, acc1 = {0.f, 0.f, 0.f, 0.f};
        u32 turns = 0;
        if (small) {
            // as little as can be is done behind X's arrival
            bf16x8 w[S::DEPTH][4], x[S::DEPTH][4];
            wait_loads(0);
#pragma unroll
            for (int e = 0; e < S::DEPTH; ++e)
                if (e < n) ds_read4(w[e], ring + behind(tail, e) * S::SLOT + w_at);
            if (TAGGED && !plain) {
                // a lane asks for its pair of every row of a chunk
                constexpr int R = XG ? CH_TAGGED_ROWS : 1;
                const int ln = fresh(lane);
                const u64* from = reinterpret_cast<const u64*>(cur.x) + (size_t)wave * rows * 64 + ln;
                u64 v[S::DEPTH][R];
                for (;;) {
                    bool late = false;
#pragma unroll
                    for (int e = 0; e < S::DEPTH; ++e)
#pragma unroll
                        for (int r = 0; r < R; ++r) {
                            const bool on = e < n && !(pair && (e & 1)) && r < (int)rows;
                            v[e][r] = on ? agent_load(from + ((size_t)(pair ? e >> 1 : e) * SW * rows + r) * 64) : pair64(0, tag);
                        }
#pragma unroll
                    for (int e = 0; e < S::DEPTH; ++e)
#pragma unroll
                        for (int r = 0; r < R; ++r) late = late || (u32)(v[e][r] >> 32) != tag;
                    if (!__any(late)) break;
                    const Args a = fresh(args);
                    if (!turn(a, ctl, turns)) return false;
                }
                // and through LDS into operands
#pragma unroll
                for (int e = 0; e < S::DEPTH; ++e)
                    if (e < n && !(pair && (e & 1)))
#pragma unroll
                        for (int r = 0; r < R; ++r)
                            asm volatile("ds_write_b32 %0, %1" ::"v"(ring + behind(tail, e) * S::SLOT + W_CHUNK + r * 256 + ln * 4), "v"((u32)v[e][r]) : "memory");
#pragma unroll
                for (int e = 0; e < S::DEPTH; ++e)
                    if (e < n && !(pair && (e & 1)))
                        ds_read_units<16>(x[e], ring + behind(tail, e) * S::SLOT + W_CHUNK + ((ln & 15) & (rows - 1)) * 256 + (ln >> 4) * 64);
            } else {
#pragma unroll
                for (int e = 0; e < S::DEPTH; ++e)
                    if (e < n && !(pair && (e & 1))) read_x(x[e], behind(tail, e), plain);
            }
#pragma unroll
            for (int e = 0; e < S::DEPTH; ++e)
                if (e < n) {
                    if (pair && (e & 1)) {
#pragma unroll
                        for (int j = 0; j < 4; ++j) acc1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[e][j], x[e & ~1][j], acc1, 0, 0, 0);
                    } else {
#pragma unroll
                        for (int j = 0; j < 4; ++j) acc0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[e][j], x[e][j], acc0, 0, 0, 0);
                    }
                }
            tail = behind(tail, n == S::DEPTH ? 0 : n);
            held = 0, pend = 0;
        } else {
            bf16x8 x[4];
            for (int e = 0; e < n; ++e) {
                const bool up = pair && (e & 1);
                bf16x8 w[4];
                wait_chunk();
                if (!up) {
                    while (read_x(x, tail, plain))
                        if (!ask_again(cur, e, turns)) return false;
                }
                ds_read4(w, ring + tail * S::SLOT + w_at);
                if (up) {
#pragma unroll
                    for (int j = 0; j < 4; ++j) acc1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[j], x[j], acc1, 0, 0, 0);
                } else {
#pragma unroll
                    for (int j = 0; j < 4; ++j) acc0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[j], x[j], acc0, 0, 0, 0);
                }
                tail = behind(tail, 1);
                --held;
                pump(seq);
            }
        }
        if (!lds_wait(ctl->summed, seq, ctl)) return false;
        put_sums(acc0, 0);
        if (pair) put_sums(acc1, 1);
        return true;
    }

    // one step of 32 keys and the state of the online softmax: attention_mfma.hip's, which has the layouts
    __device__ __forceinline__ bool attend(int seq, const Item& it) {
        const Args a = fresh(args);
        const int lane = fresh(this->lane), r16 = lane & 15, g = lane >> 4;
        const Share sh(a, ctl, it.idx);
        const int G = a->nq / a->nkv;
        is.ok = false;
        if (!lds_wait(ctl->stored, seq, ctl)) return false;
        if (sh.empty()) return lds_wait(ctl->summed, seq, ctl);
        const RL_CONSTANT ChainLayer& L = a->layers[it.layer];
        const int slot = (int)lds_get(&ctl->slot[sh.seq]);
        const int* table = a->block_table + (size_t)slot * a->table_stride;
        const u32 per_page = a->by_page.inverse;
        const int ps = a->page_size, hi = min(sh.hi, sh.pos), last = sh.pos - 1;
        const u32 stage = lds_at(lds + S::AT_STAGE);
        float m = -INFINITY, l = 0.f;
        f32x4 acc[D / 16];
#pragma unroll
        for (int b = 0; b < D / 16; ++b) acc[b] = (f32x4){0.f, 0.f, 0.f, 0.f};
        bf16x8 qf[4];
        bool first = true;
        int base = sh.lo + 32 * wave;
        while (first || base < hi) {
            bf16x8 kf[2][4], vf[D / 16];
            const bool any = base < hi;
            if (any) {
#pragma unroll
                for (int kb = 0; kb < 2; ++kb) {
                    const int key = min(base + 8 * (r16 >> 2) + 4 * kb + (r16 & 3), last);
                    const int page = (int)divide(key, per_page);
                    const bf16_t* krow = L.k_pages + (((size_t)table[page] * a->nkv + sh.hk) * ps + key - page * ps) * D;
#pragma unroll
                    for (int c = 0; c < 4; ++c) kf[kb][c] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(krow + 32 * c + 8 * g));
                }
                // (a group of eight stays inside the request's last page)
                const int key = min(base + 8 * g, last & ~7);
                const int page = (int)divide(key, per_page);
                const bf16_t* vrow = L.v_pages + (((size_t)table[page] * a->nkv + sh.hk) * D) * ps + key - page * ps;
#pragma unroll
                for (int b = 0; b < D / 16; ++b) vf[b] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(vrow + (size_t)(16 * b + r16) * ps));
            }
            if (first) {
                if (!lds_wait(ctl->ready, seq + 1, ctl)) return false;
                ds_read_row(qf, stage + min(r16, G - 1) * 256 + 16 * g);
                first = false;
            }
            if (any) {
                f32x4 s[2];
#pragma unroll
                for (int kb = 0; kb < 2; ++kb) {
                    s[kb] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int c = 0; c < 4; ++c) s[kb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[kb][c], qf[c], s[kb], 0, 0, 0);
                }
                const int seen = hi - (base + 8 * g);  // this lane's keys base + 8 g .. + 7 that are there
                float x[8];
#pragma unroll
                for (int i = 0; i < 8; ++i) x[i] = i < seen ? s[i >> 2][i & 3] * a->scale_log2 : -INFINITY;
                float mx = x[0];
#pragma unroll
                for (int i = 1; i < 8; ++i) mx = fmaxf(mx, x[i]);
                const float m_new = fmaxf(m, max_rows_of_16(mx));
                const float m_safe = m_new == -INFINITY ? 0.f : m_new;
                const float alpha = __builtin_amdgcn_exp2f(m - m_safe);
                float psum = 0.f;
                bf16x8 p;
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const float e = __builtin_amdgcn_exp2f(x[i] - m_safe);
                    psum += e;
                    p[i] = (__bf16)e;
                }
                l = l * alpha + psum;
                m = m_new;
#pragma unroll
                for (int b = 0; b < D / 16; ++b) acc[b] *= alpha;
                if (base + 32 > hi) {  // 0 * stale data must be 0
                    u32x4 mask;
#pragma unroll
                    for (int i = 0; i < 4; ++i) mask[i] = (2 * i < seen ? 0xffffu : 0u) | (2 * i + 1 < seen ? 0xffff0000u : 0u);
#pragma unroll
                    for (int b = 0; b < D / 16; ++b) vf[b] = __builtin_bit_cast(bf16x8, __builtin_bit_cast(u32x4, vf[b]) & mask);
                }
#pragma unroll
                for (int b = 0; b < D / 16; ++b) acc[b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[b], p, acc[b], 0, 0, 0);
            }
            base += CH_KEYS;
        }
        l = sum_rows_of_16(l);
        if (!lds_wait(ctl->summed, seq, ctl)) return false;
        head = tail = 0, guard = (u32)seq + 1;  // (the ring is empty)
        if (r16 < G) {
            const u32 mine = ring + S::AT_STATE;
#pragma unroll
            for (int b = 0; b < D / 16; ++b)
                asm volatile("ds_write_b128 %0, %1 offset:%2" ::"v"(mine + (r16 * D + 4 * g) * 4), "v"(acc[b]), "n"(b * 64) : "memory");
            if (g == 0)
                asm volatile("ds_write_b32 %0, %1\n ds_write_b32 %0, %2 offset:4" ::"v"(mine + (CH_MAX_GROUP * D + 2 * r16) * 4), "v"(m), "v"(l) : "memory");
        }
        return true;
    }

    __device__ __forceinline__ void run() {
        is.count = 0;
        for (int seq = 0;; ++seq) {
            const u32 t = rank + (u32)seq * workgroups;
            const Args a = fresh(args);
            if (t >= a->total) break;
            const Item it = item_of(a, t);
            if (!(it.phase == PH_ATT ? attend(seq, it) : product(seq, it))) break;
            if (lane == 0) lds_count(&ctl->streamed[0]);
        }
        stores_done();  // nothing is on its way into LDS when the wave ends
    }
};

// --------------------------------------------------------------------------------------------- //
// the wave that waits for inputs and prepares queries
// --------------------------------------------------------------------------------------------- //
template <int XG, bool TAGGED>
__device__ __forceinline__ void wait_and_prepare(Args args, unsigned char* lds, Ctl* ctl) {
    using S = Shape<XG>;
    const int lane = threadIdx.x & 63, col = lane & 15, g = lane >> 4;
    const int G = args->nq / args->nkv;
    const u32 rank = lds_get(&ctl->rank), workgroups = lds_get(&ctl->workgroups);
    const u32 tag = lds_get(&ctl->launch) + 1;
    u32 complete = 0;          // phases of the launch known to be complete
    u32 scaled = 0xffffffffu;  // the phase whose norm's factors were computed last
    for (int seq = 0;; ++seq) {
        const u32 t = rank + (u32)seq * workgroups;
        const Args a = fresh(args);
        if (t >= a->total) return;
        const Item it = item_of(a, t);
        const RL_CONSTANT ChainLayer& L = a->layers[it.layer];
        unsigned char* mine = a->space + (size_t)it.layer * a->layer_bytes;
        const u32 ph = (u32)(it.layer * PHASES + it.phase);
        // what the attention's queries need beside themselves
        const bool att = it.phase == PH_ATT;
        const bool is_q = col < G, is_k = col == G;
        f32x4 nw[4][2], cs[2][2], sn[2][2];
        if (att) {
            const int pos = Share(a, ctl, it.idx).pos;
            const float* norm = is_q ? L.q_norm : L.k_norm;
            if (norm) {
#pragma unroll
                for (int c = 0; c < 4; ++c)
#pragma unroll
                    for (int h = 0; h < 2; ++h) nw[c][h] = *reinterpret_cast<const f32x4*>(norm + 32 * c + 8 * g + 4 * h);
            }
            if (a->cos_tab) {
#pragma unroll
                for (int c = 0; c < 2; ++c)
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        const size_t at = (size_t)pos * (D / 2) + 32 * c + 8 * g + 4 * h;
                        cs[c][h] = *reinterpret_cast<const f32x4*>(a->cos_tab + at);
                        sn[c][h] = *reinterpret_cast<const f32x4*>(a->sin_tab + at);
                    }
            }
        }
        if (!TAGGED && complete < ph) {
            // every workgroup is done with the phase before
            const u64* flags = a->control->flags;
            u32 turns = 0;
            for (u32 i0 = 0; i0 < workgroups; i0 += 64 * 4) {
                bool left[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) left[j] = i0 + 64 * j + lane < workgroups;
                for (;;) {
                    u64 f[4];
#pragma unroll
                    for (int j = 0; j < 4; ++j) f[j] = left[j] ? agent_load(flags + (i0 + 64 * j + lane) * FLAG_STRIDE) : 0;
                    bool any = false;
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        left[j] = left[j] && !done_with(f[j], tag, ph);
                        any = any || left[j];
                    }
                    if (!__any(any)) break;
                    if (!turn(a, ctl, turns)) return;
                }
            }
            complete = ph;
        }
        if (!att) {
            lds_put(&ctl->ready[0], (u32)seq + 1);
            if (it.phase == PH_GU || (it.phase == PH_QKV && it.layer > 0)) {
                if (scaled != ph) {
                    // the norm's factor of every row: 64 / MP lanes add the pieces of a row's sum of squares
                    constexpr int RW = TAGGED ? CH_TAGGED_ROWS : S::MP, PER = 64 / RW;
                    const unsigned char* part = it.phase == PH_GU ? mine + a->at_part_ff : mine - a->layer_bytes + a->at_part;
                    const int parts = a->H / 16, row = lane / PER, j = lane % PER;
                    float ss = 0.f;
                    const int words = TAGGED ? parts : parts / 2;  // (an even number of pieces, two a word where it has no tag)
                    const u64* from = reinterpret_cast<const u64*>(part) + (size_t)row * words;
                    for (int p0 = 0; p0 < words; p0 += 8 * PER) {
                        u64 v[8];
                        auto at = [&](int i) { return from + p0 + i * PER + j; };
                        auto on = [&](int i) { return row < a->M && p0 + i * PER + j < words; };
                        if (TAGGED) {
                            if (!tagged(v, a, ctl, tag, at, on)) return;
#pragma unroll
                            for (int i = 0; i < 8; ++i) ss += __uint_as_float((u32)v[i]);
                        } else {
#pragma unroll
                            for (int i = 0; i < 8; ++i) v[i] = on(i) ? agent_load(at(i)) : 0;
#pragma unroll
                            for (int i = 0; i < 8; ++i) ss += __uint_as_float((u32)v[i]) + __uint_as_float((u32)(v[i] >> 32));
                        }
                    }
#pragma unroll
                    for (int o = 1; o < PER; o *= 2) ss += __shfl_xor(ss, o);
                    const float scale = rsqrtf(ss / (float)a->H + (it.phase == PH_GU ? a->ff_eps : a->norm_eps));
                    // (the factors of the item before are read: its sums have been)
                    if (!lds_wait(ctl->summed, (u32)seq, ctl)) return;
                    if (j == 0) ctl->scale[row] = scale;
                    scaled = ph;
                }
                lds_put(&ctl->scaled[0], (u32)seq + 1);
            }
            continue;
        }
        const Share sh(a, ctl, it.idx);
        if (sh.empty()) {
            lds_put(&ctl->ready[0], (u32)seq + 1);
            continue;
        }
        const int head = is_q ? sh.hk * G + col : is_k ? a->nq + sh.hk : a->nq + a->nkv + sh.hk;
        float x[4][8];
        float ss = 0.f;
        if (TAGGED) {
            u64 raw[16];
            const u64* row = reinterpret_cast<const u64*>(mine) + ((size_t)sh.seq * (a->nq + 2 * a->nkv) + head) * (D / 2);
            if (!tagged(raw, a, ctl, tag, [&](int i) { return row + 16 * (i >> 2) + 4 * g + (i & 3); }, [&](int) { return col < G + 2; })) return;
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                x[i >> 2][2 * (i & 3)] = __uint_as_float((u32)raw[i] << 16);
                x[i >> 2][2 * (i & 3) + 1] = __uint_as_float((u32)raw[i] & 0xffff0000u);
            }
        } else {
            const u64* row = reinterpret_cast<const u64*>(mine) + ((size_t)sh.seq * (a->nq + 2 * a->nkv) + head) * (D / 4);
            u64 raw[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) raw[i] = col < G + 2 ? agent_load(row + 8 * (i >> 1) + 2 * g + (i & 1)) : 0;
#pragma unroll
            for (int i = 0; i < 32; ++i) x[i >> 3][i & 7] = __uint_as_float((u32)(raw[i >> 2] >> (16 * (i & 3))) << 16);
        }
        // (attention_mfma.hip: prepared_query.  The key is one more row of the same; the value stays as it is.)
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
            for (int j = 0; j < 8; ++j) ss += x[c][j] * x[c][j];
        const float total = sum_rows_of_16(ss);
        if (col <= G) {
            if (L.q_norm) {
                const float rrms = rsqrtf(total / (float)D + a->qk_eps);
#pragma unroll
                for (int c = 0; c < 4; ++c)
#pragma unroll
                    for (int j = 0; j < 8; ++j) x[c][j] *= rrms * nw[c][j >> 2][j & 3];
            }
            if (a->cos_tab) {
#pragma unroll
                for (int c = 0; c < 2; ++c)
#pragma unroll
                    for (int j = 0; j < 8; ++j) {
                        const float p = x[c][j], q = x[c + 2][j];
                        x[c][j] = p * cs[c][j >> 2][j & 3] - q * sn[c][j >> 2][j & 3];
                        x[c + 2][j] = q * cs[c][j >> 2][j & 3] + p * sn[c][j >> 2][j & 3];
                    }
            }
        }
        // what was prepared for the item before has been read
        if (!lds_wait(ctl->summed, (u32)seq, ctl)) return;
        u32x4 y[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
#pragma unroll
            for (int j = 0; j < 4; ++j) y[c][j] = pack_bf16(x[c][2 * j], x[c][2 * j + 1]);
            if (col < G + 2) *reinterpret_cast<u32x4*>(lds + S::AT_STAGE + col * 256 + 64 * c + 16 * g) = y[c];
        }
        lds_put(&ctl->ready[0], (u32)seq + 1);
        if (sh.own()) {
            // the token's own score, of the numbers that the matrix cores would get
            float dot = 0.f;
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const u32x4 k = *reinterpret_cast<const u32x4*>(lds + S::AT_STAGE + G * 256 + 64 * c + 16 * g);
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    dot += __uint_as_float(y[c][j] << 16) * __uint_as_float(k[j] << 16);
                    dot += __uint_as_float(y[c][j] & 0xffff0000u) * __uint_as_float(k[j] & 0xffff0000u);
                }
            }
            dot = sum_rows_of_16(dot);
            if (is_q && g == 0) ctl->own[col] = dot * a->scale_log2;
            lds_put(&ctl->scaled[0], (u32)seq + 1);
            const int* table = a->block_table + (size_t)lds_get(&ctl->slot[sh.seq]) * a->table_stride;
            const int nth = (int)divide(sh.pos, a->by_page.inverse), off = sh.pos - nth * a->page_size;
            const size_t page = (size_t)table[nth] * a->nkv + sh.hk;
            if (is_k) {
                bf16_t* dst = L.k_pages + (page * a->page_size + off) * D;
#pragma unroll
                for (int c = 0; c < 4; ++c) *reinterpret_cast<u32x4*>(dst + 32 * c + 8 * g) = y[c];
            } else if (col == G + 1) {
                bf16_t* dst = L.v_pages + page * D * a->page_size + off;
#pragma unroll
                for (int c = 0; c < 4; ++c)
#pragma unroll
                    for (int j = 0; j < 8; ++j) dst[(size_t)(32 * c + 8 * g + j) * a->page_size].bits = (uint16_t)(y[c][j >> 1] >> (16 * (j & 1)));
            }
        }
    }
}

// --------------------------------------------------------------------------------------------- //
// the wave that adds and stores
// --------------------------------------------------------------------------------------------- //
// two neighbouring channels of a head, where the output product reads them
template <int XG, bool TAGGED>
__device__ __forceinline__ void store_attention(Args a, unsigned char* att, const Share& sh, int head, int lane, u32 v, u32 tag) {
    if (TAGGED)
        agent_store(reinterpret_cast<u64*>(att) + ((size_t)head * a->M + sh.seq) * 64 + lane, pair64(v, tag));
    else
        agent_store(reinterpret_cast<u32*>(att) + (((size_t)head * 16 + lane / 4) * Shape<XG>::MP + sh.seq) * 4 + lane % 4, v);
}

// The states of the waves, the token's own key and the request's other shares, folded.
template <int XG, bool TAGGED>
__device__ __forceinline__ bool fold_attention(Args a, unsigned char* lds, Ctl* ctl, const Item& it, int seq, u32 tag) {
    using S = Shape<XG>;
    const int lane = threadIdx.x & 63;
    const int G = a->nq / a->nkv;
    const Share sh(a, ctl, it.idx);
    if (sh.empty()) {
        lds_put(&ctl->summed[0], (u32)seq + 1);
        return true;
    }
    const bool own = sh.own();
    if (own && !lds_wait(ctl->scaled, (u32)seq + 1, ctl)) return false;
    const float* states = reinterpret_cast<const float*>(lds + S::AT_STATE);
    constexpr int STATE = S::RING / 4;  // numbers between two waves' states
    // lane (head, w): wave w's state of a head, w = 8 the token's own
    const int hw = lane >> 4, w = lane & 15;
    float m = -INFINITY, l = 0.f;
    if (hw < G && w < SW) m = states[w * STATE + CH_MAX_GROUP * D + 2 * hw], l = states[w * STATE + CH_MAX_GROUP * D + 2 * hw + 1];
    if (hw < G && w == SW && own) m = ctl->own[hw], l = 1.f;
    float top = m;
#pragma unroll
    for (int o = 1; o < 16; o *= 2) top = fmaxf(top, __shfl_xor(top, o));
    const float f = __builtin_amdgcn_exp2f(m - (top == -INFINITY ? 0.f : top));
    l *= f;
#pragma unroll
    for (int o = 1; o < 16; o *= 2) l += __shfl_xor(l, o);
    float o0[CH_MAX_GROUP], o1[CH_MAX_GROUP];
    auto of_lane = [](float v, int i) { return __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(v), i)); };
    const u32 v_own = own ? *reinterpret_cast<const u32*>(lds + S::AT_STAGE + (G + 1) * 256 + 4 * lane) : 0u;
#pragma unroll
    for (int h0 = 0; h0 < CH_MAX_GROUP; h0 += 2) {  // two heads' reads at a time
        if (h0 >= G) break;
        f32x2 v[2][SW];
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int i = 0; i < SW; ++i) v[h][i] = *reinterpret_cast<const f32x2*>(states + i * STATE + (h0 + h) * D + 2 * lane);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const float fo = own ? of_lane(f, 16 * (h0 + h) + SW) : 0.f;
            float p = fo * low_bf16(v_own), q = fo * high_bf16(v_own);
#pragma unroll
            for (int i = 0; i < SW; ++i) {
                const float fi = of_lane(f, 16 * (h0 + h) + i);
                p += v[h][i][0] * fi;
                q += v[h][i][1] * fi;
            }
            o0[h0 + h] = p, o1[h0 + h] = q;
        }
    }
    lds_put(&ctl->summed[0], (u32)seq + 1);
    if (sh.shares == 1) {
        unsigned char* att = a->space + (size_t)it.layer * a->layer_bytes + a->at_att;
#pragma unroll
        for (int h = 0; h < CH_MAX_GROUP; ++h) {
            if (h >= G) break;
            const float lt = of_lane(l, 16 * h);
            store_attention<XG, TAGGED>(a, att, sh, sh.hk * G + h, lane, pack_bf16(o0[h] / lt, o1[h] / lt), tag);
        }
        return true;
    }
    // The shares' states lie beside each other, a head's 128 sums, its maximum and its weight, each with the launch's number.  Where
    // every workgroup has one item of the phase at most, share s folds the heads s, s + shares, ..; else the last share, which waits
    // for items of lower numbers only, folds them all.
    const bool spread = (u32)a->n[PH_ATT] <= lds_get(&ctl->workgroups);
    const u32 share_words = (u32)a->nq * (D + 2);
    u64* states_of = a->shares + ((size_t)(it.layer * a->M + sh.seq) * a->nsplit * a->nq + sh.hk * G) * (D + 2);
    u64* mine = states_of + sh.split * share_words;
#pragma unroll
    for (int h = 0; h < CH_MAX_GROUP; ++h) {
        if (h >= G) break;
        if ((spread ? h % sh.shares : sh.shares - 1) == sh.split) continue;
        u64* to = mine + h * (D + 2);
        agent_store(to + lane, pair64(__float_as_uint(o0[h]), tag));
        agent_store(to + 64 + lane, pair64(__float_as_uint(o1[h]), tag));
        const float mh = of_lane(top, 16 * h), lh = of_lane(l, 16 * h);
        if (lane < 2) agent_store(to + D + lane, pair64(__float_as_uint(lane ? lh : mh), tag));
    }
    for (int h = 0; h < G; ++h) {
        if ((spread ? h % sh.shares : sh.shares - 1) != sh.split) continue;
        float p = 0.f, q = 0.f, lt = 0.f, mt = -INFINITY;  // in the order of the shares
        const float own_m = of_lane(top, 16 * h), own_l = of_lane(l, 16 * h);
        const float own_p = h == 0 ? o0[0] : h == 1 ? o0[1] : h == 2 ? o0[2] : o0[3], own_q = h == 0 ? o1[0] : h == 1 ? o1[1] : h == 2 ? o1[2] : o1[3];
        const u64* from = states_of + h * (D + 2);
        for (int s0 = 0; s0 < sh.shares; s0 += 8) {
            u64 v[32];
            auto on = [&](int i) { return s0 + (i >> 2) < sh.shares && s0 + (i >> 2) != sh.split; };
            auto at = [&](int i) { return from + (s0 + (i >> 2)) * share_words + ((i & 2) ? D + (i & 1) : 64 * (i & 1) + lane); };
            if (!tagged(v, a, ctl, tag, at, on)) return false;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                if (s0 + i >= sh.shares) break;
                const bool me = s0 + i == sh.split;
                const float vp = me ? own_p : __uint_as_float((u32)v[4 * i]), vq = me ? own_q : __uint_as_float((u32)v[4 * i + 1]);
                const float vm = me ? own_m : __uint_as_float((u32)v[4 * i + 2]), vl = me ? own_l : __uint_as_float((u32)v[4 * i + 3]);
                const float mn = fmaxf(mt, vm), safe = mn == -INFINITY ? 0.f : mn;
                const float keep = __builtin_amdgcn_exp2f(mt - safe), fs = __builtin_amdgcn_exp2f(vm - safe);
                lt = lt * keep + vl * fs;
                p = p * keep + vp * fs;
                q = q * keep + vq * fs;
                mt = mn;
            }
        }
        store_attention<XG, TAGGED>(a, a->space + (size_t)it.layer * a->layer_bytes + a->at_att, sh, sh.hk * G + h, lane, pack_bf16(p / lt, q / lt), tag);
    }
    return true;
}

template <int XG, bool TAGGED>
__device__ __forceinline__ void add_and_store(Args args, unsigned char* lds, Ctl* ctl) {
    using S = Shape<XG>;
    const int lane = threadIdx.x & 63, m = lane & 15, g = lane >> 4;
    const f32x4* red = reinterpret_cast<const f32x4*>(lds + S::AT_SCRATCH);
    const u32 rank = lds_get(&ctl->rank), workgroups = lds_get(&ctl->workgroups);
    const u32 tag = lds_get(&ctl->launch) + 1;
    if (!TAGGED) {  // the phases in front of its first item
        u32 done = (u32)(args->num_layers * PHASES);
        if (rank < args->total) {
            const Item it = item_of(args, rank);
            done = (u32)(it.layer * PHASES + it.phase);
        }
        if (done > 0 && lane == 0) agent_store(args->control->flags + rank * FLAG_STRIDE, pair64(done, tag));
    }
    for (int seq = 0;; ++seq) {
        const u32 t = rank + (u32)seq * workgroups;
        const Args a = fresh(args);
        if (t >= a->total) return;
        const Item it = item_of(a, t);
        const RL_CONSTANT ChainLayer& L = a->layers[it.layer];
        unsigned char* mine = a->space + (size_t)it.layer * a->layer_bytes;
        // the phases this workgroup is done with behind this item
        u32 done = (u32)(a->num_layers * PHASES);
        if (!TAGGED && t + workgroups < a->total) {
            const Item behind = item_of(a, t + workgroups);
            done = (u32)(behind.layer * PHASES + behind.phase);
        }
        const bool tells = !TAGGED && done > (u32)(it.layer * PHASES + it.phase);
        if (it.phase == PH_ATT) {
            lds_put(&ctl->stored[0], (u32)seq);
            if (!lds_wait(ctl->streamed, (u32)(SW * (seq + 1)), ctl)) return;
            if (!fold_attention<XG, TAGGED>(a, lds, ctl, it, seq, tag)) return;
        } else {
            if (!TAGGED) {
                lds_put(&ctl->stored[0], (u32)seq);
                if (!lds_wait(ctl->ready, seq + 1, ctl)) return;
            }
            const int n = it.idx * 16 + 4 * g;
            const bool row = m < a->M;
            const bool last = it.phase == PH_DOWN && L.next_norm == nullptr;
            const bool adds = (it.phase == PH_O || it.phase == PH_DOWN) && !last;
            // What the results need from memory travels while the waves multiply, and all that does not depend on them is
            // computed before they come.
            float res[4] = {0.f, 0.f, 0.f, 0.f}, nw[4] = {0.f, 0.f, 0.f, 0.f};
            const size_t at_row = (size_t)m * a->H + n;
            unsigned char *to = nullptr, *to_res = nullptr, *to_part = nullptr;  // rows of results, of the stream, pieces of sums
            if (adds) {
                const f32x4 w = *reinterpret_cast<const f32x4*>((it.phase == PH_O ? L.ff_norm : L.next_norm) + n);
                const bool streamed_in = TAGGED && !(it.phase == PH_O && it.layer == 0);  // the stream as this launch left it
                if (streamed_in) {
                    const unsigned char* from = it.phase == PH_O ? mine - a->layer_bytes + a->at_res_down : mine + a->at_res;
                    const u64* words = reinterpret_cast<const u64*>(from) + at_row;
                    u64 v[4];
                    if (!tagged(v, a, ctl, tag, [&](int i) { return words + i; }, [&](int) { return row; })) return;
#pragma unroll
                    for (int i = 0; i < 4; ++i) res[i] = __uint_as_float((u32)v[i]);
                } else if (row) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) res[i] = agent_load(a->residual + at_row + i);
                }
#pragma unroll
                for (int i = 0; i < 4; ++i) nw[i] = w[i];
                to_part = mine + (it.phase == PH_O ? a->at_part_ff : a->at_part) + ((size_t)m * (a->H / 16) + it.idx) * (TAGGED ? 8 : 4);
                to_res = TAGGED ? mine + (it.phase == PH_O ? a->at_res : a->at_res_down) + at_row * 8 : reinterpret_cast<unsigned char*>(a->residual + at_row);
            }
            if (TAGGED) lds_put(&ctl->stored[0], (u32)seq);
            if (it.phase == PH_QKV) {
                const size_t e = (size_t)m * ((a->nq + 2 * a->nkv) * D) + n;  // [row][column]
                to = mine + (TAGGED ? 4 : 2) * e;
            } else if (last) {
                to = reinterpret_cast<unsigned char*>(a->out + at_row);
            } else {
                to = mine + (it.phase == PH_GU ? a->at_act : it.phase == PH_O ? a->at_xt_ff : a->at_xt);
                if (TAGGED)  // [chunk of 128][row][pair]
                    to += (((size_t)(n / KSTEP) * a->M + m) * 64 + n % KSTEP / 2) * 8;
                else  // [group of 8][row][8]
                    to += ((size_t)(n / 8) * S::MP + m) * 16 + n % 8 * 2;
            }
            const bool tags = TAGGED && !last;
            const bool to_stream = TAGGED && it.phase == PH_O && it.layer == a->num_layers - 1;
            asm volatile("" : "+v"(to), "+v"(to_res), "+v"(to_part));
            float scale = 1.f;
            if (it.phase == PH_GU || (it.phase == PH_QKV && it.layer > 0)) {
                if (!lds_wait(ctl->scaled, (u32)seq + 1, ctl)) return;
                scale = ctl->scale[m];
            }
            if (!lds_wait(ctl->streamed, (u32)(SW * (seq + 1)), ctl)) return;
            f32x4 v = {0.f, 0.f, 0.f, 0.f}, up = {0.f, 0.f, 0.f, 0.f};
            {
                f32x4 r[SW];
                const f32x4* from = red + g * S::MP + (m & (S::MP - 1));  // (rows that are not there are stored by nobody)
#pragma unroll
                for (int w = 0; w < SW; ++w) r[w] = from[w * 8 * S::MP];
#pragma unroll
                for (int w = 0; w < SW; ++w) v += r[w];
                if (it.phase == PH_GU) {
#pragma unroll
                    for (int w = 0; w < SW; ++w) r[w] = from[(w * 2 + 1) * 4 * S::MP];
#pragma unroll
                    for (int w = 0; w < SW; ++w) up += r[w];
                }
            }
            lds_put(&ctl->summed[0], (u32)seq + 1);
            v *= scale, up *= scale;
            if (it.phase == PH_GU) {
                // (the activation reads its operands as a stored result would be)
                const u32 x0 = pack_bf16(v[0], v[1]), x1 = pack_bf16(v[2], v[3]), u0 = pack_bf16(up[0], up[1]), u1 = pack_bf16(up[2], up[3]);
                const f32x4 x = {low_bf16(x0), high_bf16(x0), low_bf16(x1), high_bf16(x1)}, u = {low_bf16(u0), high_bf16(u0), low_bf16(u1), high_bf16(u1)};
#pragma unroll
                for (int i = 0; i < 4; ++i) v[i] = x[i] / (1.f + expf(-x[i])) * u[i];
            }
            f32x4 r = {0.f, 0.f, 0.f, 0.f};
            if (adds) {
                const u32 v0 = pack_bf16(v[0], v[1]), v1 = pack_bf16(v[2], v[3]);
                r = (f32x4){res[0] + low_bf16(v0), res[1] + high_bf16(v0), res[2] + low_bf16(v1), res[3] + high_bf16(v1)};
#pragma unroll
                for (int i = 0; i < 4; ++i) v[i] = r[i] * nw[i];
            }
            const u32 p0 = pack_bf16(v[0], v[1]), p1 = pack_bf16(v[2], v[3]);
            if (row) {
                u64* at = reinterpret_cast<u64*>(to);
                if (tags) {
                    agent_store(at, pair64(p0, tag));
                    agent_store(at + 1, pair64(p1, tag));
                } else {
                    agent_store(at, pair64(p0, p1));
                }
            }
            if (adds) {
                const float sq = sum_rows_of_16(r[0] * r[0] + r[1] * r[1] + r[2] * r[2] + r[3] * r[3]);
                if (row && g == 0) {
                    if (TAGGED)
                        agent_store(reinterpret_cast<u64*>(to_part), pair64(__float_as_uint(sq), tag));
                    else
                        agent_store(reinterpret_cast<float*>(to_part), sq);
                }
                if (row) {
                    u64* at = reinterpret_cast<u64*>(to_res);
                    if (TAGGED) {
#pragma unroll
                        for (int i = 0; i < 4; ++i) agent_store(at + i, pair64(__float_as_uint(r[i]), tag));
                    }
                    if (to_stream) at = reinterpret_cast<u64*>(a->residual + at_row);  // (what follows the launch reads it there)
                    if (!TAGGED || to_stream) {
                        agent_store(at, pair64(__float_as_uint(r[0]), __float_as_uint(r[1])));
                        agent_store(at + 1, pair64(__float_as_uint(r[2]), __float_as_uint(r[3])));
                    }
                }
            }
        }
        if (tells) {
            stores_done();
            if (lane == 0) agent_store(a->control->flags + rank * FLAG_STRIDE, pair64(done, tag));
        }
    }
}

template <int XG, bool TAGGED>
__global__ __launch_bounds__(CH_THREADS) void decode_chain_kernel(ChainArgs) {
    using S = Shape<XG>;
    const Args a = (Args)__builtin_amdgcn_kernarg_segment_ptr();
    __shared__ __attribute__((aligned(1024))) unsigned char lds[S::BYTES];
    static_assert(sizeof(Ctl) <= S::CTL && S::BYTES <= 160 * 1024, "LDS");
    Ctl* ctl = reinterpret_cast<Ctl*>(lds + S::AT_CTL);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / RL_WAVE);
    Control* control = a->control;
    if (threadIdx.x == 0) {
        const u32 launch = agent_load(&control->launch), given_up = agent_load(&control->abort);
        const u32 rank = __hip_atomic_fetch_add(&control->list, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        u32 workgroups = 0;
        if (rank == 0) {
            for (u32 turns = 0; agent_load(&control->list) < gridDim.x && turns < LIST_TURNS; ++turns) __builtin_amdgcn_s_sleep(1);
            workgroups = __hip_atomic_fetch_or(&control->list, LIST_CLOSED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            agent_store(&control->dealt, pair64(workgroups, launch + 1));
        } else if (!(rank & LIST_CLOSED)) {
            for (u32 turns = 0; turns < FLAG_TURNS; ++turns) {
                const u64 dealt = agent_load(&control->dealt);
                if ((u32)(dealt >> 32) == launch + 1) {
                    workgroups = (u32)dealt;
                    break;
                }
            }
        }
        const u32 over = given_up || (!(rank & LIST_CLOSED) && workgroups == 0);
        ctl->rank = over || workgroups == 0 ? 0xffffffffu : rank;  // (or too late for the list)
        ctl->workgroups = workgroups;
        ctl->launch = launch;
        ctl->ready[0] = ctl->summed[0] = ctl->streamed[0] = ctl->scaled[0] = ctl->stored[0] = 0;
        ctl->ready[1] = ctl->summed[1] = ctl->streamed[1] = ctl->scaled[1] = ctl->stored[1] = over;
    }
    if (threadIdx.x < (u32)a->M) {
        const int pos = a->positions[threadIdx.x], kend = pos + 1;
        int run = ((kend + a->nsplit - 1) / a->nsplit + 31) & ~31;
        run = kend <= CH_ALONE ? CH_ALONE : max(run, CH_KEYS);
        ctl->pos[threadIdx.x] = pos;
        ctl->slot[threadIdx.x] = a->token_slot[threadIdx.x];
        ctl->run[threadIdx.x] = run;
        ctl->shares[threadIdx.x] = (kend + run - 1) / run;
    }
    __syncthreads();
    if (lds_get(&ctl->rank) != 0xffffffffu) {
        if (wave < SW)
            Streamer<XG, TAGGED>(a, lds, ctl, wave).run();
        else if (wave == SW)
            wait_and_prepare<XG, TAGGED>(a, lds, ctl);
        else
            add_and_store<XG, TAGGED>(a, lds, ctl);
    }
    __syncthreads();
    if (lds_get(&ctl->ready[1])) {  // a wait ran into its bound
        for (size_t i = threadIdx.x; i < (size_t)a->M * a->H; i += CH_THREADS) a->out[i].bits = 0x7fc0;
        if (threadIdx.x == 0) {
            agent_store(&control->abort, 1u);
            __hip_atomic_store(a->notice, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        }
    }
    const u32 launch = lds_get(&ctl->launch);
    if (launch == LAST_LAUNCH) {  // what any wave has stored is there before somebody clears it
        stores_done();
        __syncthreads();
    }
    u32 last = 0;
    if (threadIdx.x == 0) {
        stores_done();
        const u32 before = __hip_atomic_fetch_add(&control->left, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        last = before + 1 == gridDim.x;
        if (last) {  // as the next launch wants to find it
            agent_store(&control->list, 0u);
            agent_store(&control->left, 0u);
            agent_store(&control->launch, launch == LAST_LAUNCH ? 0u : launch + 1);
        }
    }
    if (launch != LAST_LAUNCH) return;
    if (threadIdx.x == 0) ctl->rank = last;
    __syncthreads();
    if (!lds_get(&ctl->rank)) return;
    for (u64 i = threadIdx.x; i < a->tagged_words; i += CH_THREADS) agent_store(a->tagged + i, (u64)0);
    for (u64 i = threadIdx.x; i < a->share_words; i += CH_THREADS) agent_store(a->shares + i, (u64)0);
    for (u32 i = threadIdx.x; i < CH_MAX_WORKGROUPS * FLAG_STRIDE; i += CH_THREADS) agent_store(control->flags + i, (u64)0);
    if (threadIdx.x == 0) agent_store(&control->dealt, (u64)0);
}

// a layer's space; tagged results have a part of the space of their own, so that what lies in a number's place is always
// an earlier launch's
static long long lay_out(ChainArgs& a, int rows, int hidden, int nq, int nkv, int inter) {
    const bool tags = rows <= CH_TAGGED_ROWS;
    const long long mp = rows <= 4 ? 4 : rows <= 8 ? 8 : 16;
    long long at = 0;
    auto room = [&](long long bytes) {
        const long long here = at;
        at += (bytes + 255) / 256 * 256;
        return (u32)here;
    };
    const long long e = tags ? 4ll * CH_TAGGED_ROWS : 2ll * mp;  // bytes of a column of rows
    room((nq + 2ll * nkv) * D * e);
    a.at_att = room((long long)nq * D * e);
    a.at_xt_ff = room(hidden * e);
    a.at_part_ff = room(hidden / 16 * (tags ? 8ll : 4ll) * mp);
    a.at_act = room(inter * e);
    a.at_xt = room(hidden * e);
    a.at_part = room(hidden / 16 * (tags ? 8ll : 4ll) * mp);
    a.at_res = tags ? room(hidden * 8ll * CH_TAGGED_ROWS) : 0;
    a.at_res_down = tags ? room(hidden * 8ll * CH_TAGGED_ROWS) : 0;
    a.layer_bytes = (u32)at;
    return at;
}

static long long items_of_layer(ChainArgs& a, int rows, int hidden, int nq, int nkv, int inter, int nsplit) {
    const long long shares = (long long)rows * nkv * nsplit;
    a.n[PH_QKV] = (nq + 2 * nkv) * (D / 16), a.n[PH_ATT] = (int)shares, a.n[PH_O] = a.n[PH_DOWN] = hidden / 16, a.n[PH_GU] = inter / 16;
    return (nq + 2ll * nkv) * (D / 16) + shares + 2 * (hidden / 16) + inter / 16;
}

extern "C" int rl_decode_chain_layer_bytes() { return (int)sizeof(ChainLayer); }
extern "C" int rl_decode_chain_max_group() { return CH_MAX_GROUP; }
extern "C" int rl_decode_chain_min_keys() { return CH_KEYS; }
extern "C" int rl_decode_chain_control() { return (int)sizeof(Control); }
extern "C" int rl_decode_chain_launch_word() { return (int)offsetof(Control, launch); }
extern "C" int rl_decode_chain_abort_word() { return (int)offsetof(Control, abort); }
// Where the device finds a word of pinned host memory.
extern "C" int rl_decode_chain_notice(void* host, void** device) {
    return hipHostGetDevicePointer(device, host, 0) == hipSuccess ? RL_OK : RL_ERR_ARG;
}
extern "C" unsigned rl_decode_chain_last_launch() { return LAST_LAUNCH; }
// (the waits' comparison, of launch number `launch`)
extern "C" int rl_decode_chain_done(unsigned long long flag, unsigned launch, unsigned phases) { return done_with(flag, launch + 1, phases); }

// Bytes for steps of these sizes: of rows, and of the attention's shares.
extern "C" long long rl_decode_chain_space(int num_layers, int rows, int hidden, int nq, int nkv, int inter) {
    ChainArgs a;
    return lay_out(a, rows, hidden, nq, nkv, inter) * num_layers;
}
extern "C" long long rl_decode_chain_shares(int num_layers, int rows, int nq, int nsplit) {
    return nsplit < 2 ? 0 : 8ll * num_layers * rows * nsplit * nq * (D + 2);
}

// Whether the launch takes layers, steps and a cache of these sizes.  (The last line: every index is divided by a
// multiplication, which is exact below 2^32 / divisor.)
extern "C" int rl_decode_chain_takes(int num_layers, int rows, int hidden, int nq, int nkv, int inter, int table_stride,
                                     int page_size, int nsplit, int units) {
    if (num_layers < 1 || rows < 1 || rows > CH_MAX_ROWS || nkv < 1 || nq % nkv || nq / nkv > CH_MAX_GROUP) return 0;
    if (hidden % KSTEP || inter % KSTEP || hidden < KSTEP || inter < KSTEP || page_size < 8 || page_size % 8) return 0;
    if (nsplit < 1 || units < 1 || units > CH_MAX_WORKGROUPS || table_stride < 1) return 0;
    ChainArgs a;
    const long long per_layer = items_of_layer(a, rows, hidden, nq, nkv, inter, nsplit);
    if (lay_out(a, rows, hidden, nq, nkv, inter) > 0x7fffffffll || per_layer * num_layers + units > 0x7fffffffll) return 0;
    return (u64)(per_layer * num_layers + units) * per_layer < 0x100000000ull && (u64)table_stride * page_size * page_size < 0x100000000ull;
}

// `tagged_space`, `space`, `shares`: as large as the two functions above say for up to CH_TAGGED_ROWS rows, for more, and for all.
// `control` and the two that hold tags, of `tagged_bytes` and `shares_bytes`, are zeros before the first launch; launches that share
// them follow each other.  `notice`: rl_decode_chain_notice's.
extern "C" int rl_decode_chain(const void* layers, const void* x, float* residual, void* out, const int* positions,
                               const int* token_slot, const int* block_table, const float* cos_tab, const float* sin_tab,
                               void* tagged_space, long long tagged_bytes, void* space, void* shares, long long shares_bytes,
                               void* control, void* notice, int num_layers, int rows, int hidden,
                               int nq, int nkv, int inter, int table_stride, int page_size, int nsplit, float scale, float qk_eps,
                               float norm_eps, float ff_eps, int units, hipStream_t stream) {
    if (!rl_decode_chain_takes(num_layers, rows, hidden, nq, nkv, inter, table_stride, page_size, nsplit, units)) return RL_ERR_ARG;
    if (tagged_bytes < 0 || shares_bytes < 0 || !notice || (cos_tab != nullptr) != (sin_tab != nullptr)) return RL_ERR_ARG;
    ChainArgs a;
    lay_out(a, rows, hidden, nq, nkv, inter);
    const long long per_layer = items_of_layer(a, rows, hidden, nq, nkv, inter, nsplit);
    a.layers = (const RL_CONSTANT ChainLayer*)layers;
    a.x = (const bf16_t*)x, a.residual = residual, a.out = (bf16_t*)out;
    a.positions = positions, a.token_slot = token_slot, a.block_table = block_table;
    a.cos_tab = cos_tab, a.sin_tab = sin_tab;
    a.space = (unsigned char*)(rows <= CH_TAGGED_ROWS ? tagged_space : space);
    a.shares = (u64*)shares;
    a.control = (Control*)control;
    a.tagged = (u64*)tagged_space, a.tagged_words = tagged_bytes / 8, a.share_words = shares_bytes / 8;
    a.notice = (u32*)notice;
    a.num_layers = num_layers, a.M = rows, a.H = hidden, a.nq = nq, a.nkv = nkv, a.I = inter;
    a.table_stride = table_stride, a.page_size = page_size, a.nsplit = nsplit;
    a.scale_log2 = scale * 1.4426950408889634f, a.qk_eps = qk_eps, a.norm_eps = norm_eps, a.ff_eps = ff_eps;
    a.per_layer.set((u32)per_layer), a.by_heads.set(nkv), a.by_rows.set(rows), a.by_page.set(page_size);
    a.total = (u32)(per_layer * num_layers);
#define RL_CHAIN(XG, TAGGED) hipLaunchKernelGGL((decode_chain_kernel<XG, TAGGED>), dim3(units), dim3(CH_THREADS), 0, stream, a)
    if (rows == 1)
        RL_CHAIN(0, true);
    else if (rows <= CH_TAGGED_ROWS)
        RL_CHAIN(1, true);
    else if (rows <= 4)
        RL_CHAIN(1, false);
    else if (rows <= 8)
        RL_CHAIN(2, false);
    else
        RL_CHAIN(4, false);
#undef RL_CHAIN
    return rl_launch_status();
}
