// Which element a draw picks: the first at which the running sum of the probabilities reaches the target, the walk being shared among threads that each have a
// run of elements.  A thread knows the running sum in front of its run (`lower`) and behind it (`end`), both rounded; one thread's end is the next one's lower,
// the same number, so that no target lies between two threads.
#pragma once

#include <hip/hip_runtime.h>

// The first thread whose run this holds for takes the draw, or, where rounding leaves the target above every end, the last one whose run has any weight.  (A
// run without weight is never asked: its end may be a last bit above that of the run before it.)
__host__ __device__ inline bool draw_reaches(double own, double end, double target) { return own > 0.0 && target <= end; }

// That thread's walk over its elements: the first that reaches the target, or the last that has any weight
struct DrawWalk {
    double sum, target;  // at first: lower
    int pick = 0;
    bool there = false;
    __host__ __device__ DrawWalk(double lower, double target) : sum(lower), target(target) {}
    __host__ __device__ void next(int i, float p) {
        if (there || !(p > 0.0f)) return;
        sum += (double)p;
        pick = i;
        there = sum >= target;
    }
};
