// bx_runs.h -- when fused steps may be taken in runs (bx_capi.hip,
// fused_loop).  Integers only.
#pragma once

namespace bx {

constexpr int kChunkSteps = 32;             // steps per run, at most
constexpr int kCalmSteps = 8 * kChunkSteps;

// A run in which a step meets an irregular branch is undone as a whole and its
// steps are taken one at a time, at least one run's worth, as after any
// irregular step.  Each undone run doubles that pause, up to kCalmSteps, until
// so many regular steps have followed one another: irregular steps that keep
// coming then waste no more than an eighth of the steps taken (with the same
// pause each time, one in every 40 to 64 steps nearly doubled the work), while
// a flow with a few of them, or with all of them in a row, resumes its runs at
// once.  (Short runs in place of the pause cost more than they save: 128^3
// cells with one irregular step in 400, 253 us per step, 259 with runs of an
// eighth of the regular steps so far.)
struct RunPacing {
    int pause = 0;               // steps to take one at a time before the next run
    int next = kChunkSteps;      // the pause after the next undone run
    int calm = kCalmSteps;       // regular steps since the last irregular one, counted up to here
    bool may_run() const { return pause == 0; }
    void regular(int steps)
    {
        pause = pause > steps ? pause - steps : 0;
        calm = calm + steps < kCalmSteps ? calm + steps : kCalmSteps;
        if (calm == kCalmSteps) next = kChunkSteps;
    }
    void undone()
    {
        pause = next;
        next = 2 * next < kCalmSteps ? 2 * next : kCalmSteps;
        calm = 0;
    }
    void irregular()
    {
        pause = pause > kChunkSteps ? pause - 1 : kChunkSteps;
        calm = 0;
    }
};

}  // namespace bx
