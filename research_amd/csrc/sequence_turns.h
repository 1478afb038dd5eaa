// In which order the workgroups of a prompt kernel take the sequences of a batch.  Plain C++, shared with the CPU tests.
#pragma once
#include <stdint.h>

#if defined(__HIPCC__)
#define PA_TURN_FN __host__ __device__ inline __attribute__((always_inline))
#else
#define PA_TURN_FN inline
#endif

// Workgroups go to the eight dies in the order of their ids, inside a die to groups of compute units in turn, and wait for the one
// whose turn it is: a sequence whose workgroups always came to the same places would keep the others waiting.  The sequence that
// index `x` of `batch` stands for in turn `turn` (a block of rows): one further every turn moves it over the dies, one more every
// eight turns over the groups inside a die.
PA_TURN_FN int sequence_in_turn(int x, int turn, int batch) { return (int)((uint32_t)(x + turn + (turn >> 3)) % (uint32_t)batch); }
