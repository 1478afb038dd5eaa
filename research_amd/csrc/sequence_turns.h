// In which order the workgroups of a prompt kernel take the sequences of a batch.  Plain C++, shared with the CPU tests.
#pragma once
#include <stdint.h>

#if defined(__HIPCC__)
#define PA_TURN_FN __host__ __device__ inline __attribute__((always_inline))
#else
#define PA_TURN_FN inline
#endif

// Workgroups go to the eight dies in the order of their ids, inside a die to four groups of compute units in turn, and wait for the
// one whose turn it is: a sequence whose workgroups always came to the same places would keep the others waiting.  The sequence that
// index `x` of `batch` stands for in turn `turn` (a block of rows): one further every turn moves it over the dies; with `inside`, one
// more every eight turns also over the groups inside a die.
PA_TURN_FN int sequence_in_turn(int x, int turn, int batch, bool inside) {
    return (int)((uint32_t)(x + turn + (inside ? turn >> 3 : 0)) % (uint32_t)batch);
}
// Whether it needs that: `side` workgroups of a sequence and turn have neighbouring ids.  Where a turn's ids fill all 32 places (8
// sequences over four heads of keys) the turns alone spread it.
PA_TURN_FN bool turns_miss_groups(int side, int batch) { return (int64_t)side * batch % 32 != 0; }
