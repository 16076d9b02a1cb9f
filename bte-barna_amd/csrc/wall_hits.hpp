// The hit counters of a wall.
#pragma once
#include <stdint.h>

namespace bte {

// Takes the signed hits of one side out of its counters: those of the step
// and source kernels (step_hits) and of the emission before (emit_hits), and
// clears the first and the word that the emission after next will count in.
// Every wave of the workgroup calls it and gets the same sum. The two parts
// may cancel, so the sum alone does not say that both words are zero:
// all_read, a barrier of the workgroup, stands between the last wave's reads
// and the clearing by one thread (clears), whatever the sum is.
template <class Barrier>
__device__ __host__ inline int take_wall_hits(int32_t* step_hits, const int32_t* emit_hits, int32_t* later_hits,
                                              bool clears, Barrier all_read) {
    const int E = *step_hits + *emit_hits;
    all_read();
    if (clears) {
        *step_hits = 0;
        *later_hits = 0;
    }
    return E;
}

}  // namespace bte
