// take_wall_hits by the waves of a workgroup, each run up to its barrier
// before the next one begins (the barrier of wave w runs the waves after it),
// so that a word cleared without a barrier is seen by all later waves
#include <cstdio>
#include <cstdlib>
#include "wall_hits.hpp"
static const int WAVES = 4;
static int32_t step_hits, emit_hits, later_hits;
static int got[WAVES], started;
static void wave(int w) {
    if (w == WAVES || started > w) return;
    started = w + 1;
    got[w] = bte::take_wall_hits(&step_hits, &emit_hits, &later_hits, w == 0, [w] { wave(w + 1); });
    wave(w + 1);
}
int main() {
    const int hits[][2] = {{0, 0}, {5, -5}, {-1, 1}, {7, 2}, {-3, -4}, {0, 6}, {6, 0}};
    for (auto& h : hits) {
        step_hits = h[0], emit_hits = h[1], later_hits = 9, started = 0;
        wave(0);
        for (int w = 0; w < WAVES; w++)
            if (got[w] != h[0] + h[1]) return printf("hits %d %d: wave %d takes %d\n", h[0], h[1], w, got[w]), 1;
        if (step_hits != 0 || later_hits != 0 || emit_hits != h[1]) return printf("hits %d %d: not cleared\n", h[0], h[1]), 1;
    }
    printf("ok\n");
}
