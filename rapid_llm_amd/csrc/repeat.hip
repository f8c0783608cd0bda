// The launches of one layer, made again for the layers behind it without a trip through the caller's
// language: every entry point of this package takes pointers and integers and a few floats and returns a
// code, so a call is an address and two lists.  What differs between layers are pointers, which come out of a table.
//
// A launch made from Python costs the host 11 to 13 us (checks, conversions, the call), one made here 2.6: a prompt
// step of the smallest model, 8 launches a layer of 3 to 12 us each, was bound by the host.
#include "common.h"

#define RL_CALL_INTS 32
#define RL_CALL_FLOATS 8

struct RlCall {
    void* entry;
    long long ints[RL_CALL_INTS];  // pointers and integers, in their order
    float floats[RL_CALL_FLOATS];  // floats, in theirs
};

// argument `arg` of call `call` is the pointer in `column` of row (place - back) of the table
struct RlSlot {
    int call, arg, column, back;
};

#if defined(__x86_64__) && defined(__linux__)
// System V AMD64 calling convention: integers and pointers go to six registers and then, eight bytes each, to the
// stack in their order, floats to eight registers of their own (no more are passed here); the callee reads as many
// of each as it has and the caller clears the stack, so one type serves every signature.
typedef long long I;
typedef int (*RlEntry)(I, I, I, I, I, I, I, I, I, I, I, I, I, I, I, I, I, I, I, I, I, I, I, I, I, I, I, I, I, I, I, I, float, float,
                       float, float, float, float, float, float);

// what a call holds at most, 0 on hosts whose calls are not known here
extern "C" int rl_repeat_max_ints() { return RL_CALL_INTS; }
extern "C" int rl_repeat_max_floats() { return RL_CALL_FLOATS; }

static int make_call(const RlCall& c) {
    const long long* i = c.ints;
    const float* f = c.floats;
    return ((RlEntry)c.entry)(i[0], i[1], i[2], i[3], i[4], i[5], i[6], i[7], i[8], i[9], i[10], i[11], i[12], i[13], i[14],
                              i[15], i[16], i[17], i[18], i[19], i[20], i[21], i[22], i[23], i[24], i[25], i[26], i[27], i[28],
                              i[29], i[30], i[31], f[0], f[1], f[2], f[3], f[4], f[5], f[6], f[7]);
}
#else
extern "C" int rl_repeat_max_ints() { return 0; }
extern "C" int rl_repeat_max_floats() { return 0; }

static int make_call(const RlCall&) { return RL_ERR_ARG; }
#endif

// The calls in their order for the places first .. last - 1; returns the first code that is not 0 (nothing behind
// it is made).  The calls' slots are overwritten.
extern "C" int rl_repeat_calls(RlCall* calls, int num_calls, const RlSlot* slots, int num_slots, const long long* table,
                               int columns, int first, int last) {
    for (int s = 0; s < num_slots; ++s)
        if (slots[s].call < 0 || slots[s].call >= num_calls || slots[s].arg < 0 || slots[s].arg >= RL_CALL_INTS ||
            slots[s].column < 0 || slots[s].column >= columns || slots[s].back < 0 || slots[s].back > first)
            return RL_ERR_ARG;
    for (int place = first; place < last; ++place) {
        for (int s = 0; s < num_slots; ++s)
            calls[slots[s].call].ints[slots[s].arg] = table[(long long)(place - slots[s].back) * columns + slots[s].column];
        for (int c = 0; c < num_calls; ++c) {
            const int code = make_call(calls[c]);
            if (code != RL_OK) return code;
        }
    }
    return RL_OK;
}
