// Status of a chain of launches that run as steps a = 0, 1, ... in stream
// order: step a reads word a and writes word a + 1, so no launch reads a word
// that it writes, and every wave of every workgroup of a step, however late it
// starts, finds the same word (with one word for all steps, waves of one
// workgroup could disagree on the step that stops, and part of them go on past
// barriers that the others never reach).  All words start as STEP_RUNNING; one
// thread of the step stores.
#pragma once
#ifdef __HIPCC__
#define STEP_FN __host__ __device__ __forceinline__
#else
#define STEP_FN inline
#endif

namespace mcmb {

constexpr int STEP_RUNNING = -1;

// words of a chain whose last step is amax
STEP_FN int step_words(int amax) { return amax + 2; }
STEP_FN int step_status(const int* st, int a) { return st[a]; }
// the chain stops with code at step a; a step that finds it stopped passes its
// status on
STEP_FN void step_stop(int* st, int a, int code) { st[a + 1] = code; }

}  // namespace mcmb
